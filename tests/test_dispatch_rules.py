"""The host's kernel choice at both sides of its rules, through attn_flash_plan: nothing is launched
and no tensor exists, so shapes of any size can be asked for."""
import pytest

import transfer_station_amd as ts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _full_mi355x():
    assert ts.device_count() >= 1, "no HIP device visible: GPU tests must run on the MI355X box"
    if ts.device_info()["cus"] != 256:
        pytest.skip("the kernel choice is pinned for a 256-CU MI355X")


def plan(Hq, Hkv, Sq, Sk, D, causal, vt=0):
    p = ts.attn_flash_plan(Hq, Hkv, Sq, Sk, D, causal, 128, vt)
    print("plan", (Hq, Hkv, Sq, Sk, D, causal, vt), p, flush=True)
    return p


@pytest.mark.parametrize("Hq,Hkv,S,D", [
    (64, 16, 20000, 256),    # the loads compared stay below 2^31
    (64, 16, 55000, 256),    # three loads of 4-wave tiles pass 2^31
    (192, 48, 32768, 256),
    (192, 48, 32768, 192),
    (1024, 128, 100000, 256),  # one load passes 2^32
])
def test_long_causal_wide_heads_take_8_waves(Hq, Hkv, S, D):
    """Causal grids of thousands of tiles at D > 128: the tile loads that the rule compares need 64
    bits."""
    name = plan(Hq, Hkv, S, S, D, 1)[0][0]
    assert name.startswith("attn_prefill_fast_kernel<%d, %d, 8, " % (D, 32 if D == 256 else 64))


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, V^T, row blocks per workgroup, grid, parts
    (2048, 32, 1, 4001, 128, 0, 2, 512, 8),    # four blocks of 16 rows
    (1536, 32, 1, 4001, 128, 0, 2, 512, 8),    # three
    (1024, 32, 1, 4001, 128, 0, 1, 512, 8),    # two: one each
    (2048, 32, 1, 4001, 160, 0, 1, 512, 4),    # D > 128
    (2048, 32, 1, 4000, 128, 1, 2, 512, 8),
    # few kv heads: the grid that is launched, after the cap of 64 parts, has a workgroup per CU
    (64, 1, 1, 65536, 64, 0, 1, 512, 128),
    (64, 1, 1, 32768, 128, 0, 1, 512, 128),
    (64, 1, 1, 16500, 40, 0, 1, 260, 65),
    (128, 2, 1, 32768, 128, 0, 2, 256, 64),
    (48, 3, 3, 65536, 128, 0, 2, 384, 64),
    # 96 KB of K and V per workgroup (two 128-key steps at D = 128, three at 64)
    (4096, 64, 1, 500, 128, 0, 1, 512, 2),
    (4096, 64, 1, 1000, 128, 0, 2, 512, 4),
    (4096, 64, 1, 1000, 64, 0, 1, 512, 2),
    (256, 4, 1, 16500, 64, 0, 2, 344, 43),
    # 256 KB where one block per workgroup needs no parts
    (1600, 200, 6, 500, 64, 0, 1, 600, 1),
    (8192, 128, 1, 1000, 64, 0, 1, 512, 1),
    (8192, 128, 1, 2000, 64, 0, 2, 512, 2),
    (8192, 128, 1, 1000, 128, 0, 2, 512, 2),
])
def test_decode_row_blocks_per_workgroup(case):
    Hq, Hkv, Sq, Sk, D, vt, blocks, grid, parts = case
    p = plan(Hq, Hkv, Sq, Sk, D, Sq > 1, vt)
    name, notes, g = p[0][:3]
    assert name.startswith("attn_decode_"), case
    assert (2 if ", 2 blocks" in name else 1) == blocks, case
    assert int(g) == grid and "nsplit=%d" % parts in notes.split(), case
    assert len(p) == (1 if parts == 1 else 2), case


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, causal, V^T, what the first kernel's name starts with
    # V^T decode: one-step parts straight from memory, longer ones staged (unaligned: from 3 steps)
    (32, 8, 1, 776, 128, 0, 1, "attn_decode_kernel<128, false, true, true, "),
    (256, 64, 1, 1024, 128, 0, 1, "attn_decode_kernel<128, false, true, true, "),
    (256, 64, 1, 1032, 128, 0, 1, "attn_decode_vt_kernel<128, false, "),
    (512, 128, 1, 1025, 128, 0, 1, "attn_decode_vt_kernel<128, false, "),
    (512, 128, 1, 1001, 128, 0, 1, "attn_decode_kernel<128, false, false, true, "),
    (64, 64, 1, 3001, 256, 0, 1, "attn_decode_kernel<256, false, false, true, "),
    # head dims past 128: 192-wide and 256-wide tiles, 8 and 4 waves
    (64, 16, 2048, 2048, 192, 0, 0, "attn_prefill_fast_kernel<192, 64, 8, "),
    (64, 16, 2048, 2048, 200, 0, 0, "attn_prefill_fast_kernel<256, 32, 8, "),
    (64, 16, 2048, 2048, 256, 1, 0, "attn_prefill_fast_kernel<256, 32, 8, "),
    (24, 8, 2048, 2048, 256, 1, 0, "attn_prefill_fast_kernel<256, 64, 4, "),
    (32, 8, 1000, 1000, 136, 0, 0, "attn_prefill_fast_kernel<192, 64, 4, "),
    # without the vector layout
    (24, 6, 1000, 2003, 100, 0, 0, "attn_prefill_fast_kernel<128, 128, 8, false, false, true, unal"),
    (64, 16, 2048, 2003, 128, 0, 1, "attn_prefill_fast_kernel<128, 64, 8, false, true, false, unal"),
    (64, 16, 2048, 2048, 250, 0, 0, "attn_prefill_fast_kernel<256, 32, 8, false, false, false, unal"),
    (8, 2, 100, 2048, 250, 0, 0, "attn_prefill_fast_kernel<256, 32, 4, false, false, false, unal"),
    (8, 2, 100, 2048, 7, 0, 0, "attn_prefill_fast_kernel<64, 128, 4, false, false, false, unal"),
])
def test_kernels_by_shape(case):
    Hq, Hkv, Sq, Sk, D, causal, vt, want = case
    assert plan(Hq, Hkv, Sq, Sk, D, causal, vt)[0][0].startswith(want), case


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, two workgroups per CU instead of three
    (1600, 400, 1, 3560, 96, 1),    # 800 workgroups: 3 per CU would leave a round of 32
    (1600, 400, 1, 3560, 99, 1),    # without the vector layout
    (1600, 400, 1, 2047, 96, 1),    # 1024 keys each
    (1600, 400, 1, 1792, 96, 0),    # 896 keys each
    (1536, 384, 1, 3560, 128, 0),   # 768: three full per CU
    (2048, 512, 1, 4096, 128, 0),
    (3200, 800, 1, 3560, 128, 1),   # unsplit
    (6400, 1600, 1, 3560, 128, 0),  # 1600: no better filled by twos
    (1600, 400, 1, 3560, 64, 0),    # other instances
    (1600, 400, 1, 3560, 160, 0),
])
def test_decode_rounds_of_two_per_cu(case):
    Hq, Hkv, Sq, Sk, D, two = case
    assert ("two-per-cu=1" in plan(Hq, Hkv, Sq, Sk, D, 0)[0][1].split()) == bool(two), case
