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
