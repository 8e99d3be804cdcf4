"""Tensors without the 16-byte vector layout: head dims that are no multiple of 8, V^T rows of an
odd key count, bases at any element. The kernels read such rows 16 bytes at a time, the pieces at a
row's end as its last eight elements; each case here ends rows, tiles or tensors inside a piece.
Inputs lie between NaN guards (a value taken from outside a tensor makes the output NaN) and O
between guards that must survive."""
import numpy as np
import pytest

import transfer_station_amd as ts

pytestmark = pytest.mark.gpu

PAD = 32  # guard elements on each side


@pytest.fixture(scope="module", autouse=True)
def _gpu_present():
    assert ts.device_count() >= 1, "no HIP device visible: GPU tests must run on the MI355X box"


def guarded(arr, off):
    """(buffer, address of arr's copy in it), off elements past a 16-byte boundary."""
    full = np.full(arr.size + 2 * PAD + off, 0xFFFF, np.uint16)
    full[PAD + off:PAD + off + arr.size] = arr
    buf = ts.DeviceBuffer.from_array(full)
    return buf, buf.ptr + 2 * (PAD + off)


def attend(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, vt, off):
    n = Hq * Sq * D
    bufs = [guarded(a, off) for a in (Q, K, V)]
    with ts.DeviceBuffer(4 * (n + 2 * PAD)) as do, \
            ts.DeviceBuffer(ts.attn_flash_scratch_bytes(D, 128)) as ds:
        do.fill_bytes(0xFF)
        ds.fill_bytes(0xFF)
        ts.attn_flash(bufs[0][1], bufs[1][1], bufs[2][1], do.ptr + 4 * PAD, Hq, Hkv, Sq, Sk, D,
                      causal, 128, ds, vt)
        ts.synchronize()
        raw = do.download(np.uint32)
    for b, _ in bufs:
        b.free()
    assert np.all(raw[:PAD] == 0xFFFFFFFF) and np.all(raw[PAD + n:] == 0xFFFFFFFF)
    return raw[PAD:PAD + n].view(np.float32)


CASES = [
    # Hq, Hkv, Sq, Sk, D, causal, base offset in elements
    (4, 2, 70, 65, 7, 1, 0),          # rows shorter than a piece
    (4, 2, 70, 129, 9, 0, 0),         # one whole piece and one element
    (6, 3, 130, 257, 65, 1, 0),       # 96-wide tiles, key halves, a one-key last tile
    (8, 2, 200, 1023, 100, 0, 0),     # key split: partials of a head dim that is no multiple of 8
    (8, 2, 500, 501, 127, 1, 0),      # causal key split at DP = 128
    (160, 40, 300, 255, 100, 0, 0),   # 8 waves, ragged query and key tails
    (136, 34, 520, 521, 81, 1, 0),    # 8 waves, causal, DP = 96
    (40, 40, 1000, 70, 63, 1, 0),     # Sq > Sk: rows that attend nothing
    (32, 8, 20, 333, 44, 1, 0),       # packed short query blocks
    (4, 2, 140, 100, 129, 1, 0),      # 256-wide tiles
    (2, 1, 33, 63, 255, 0, 0),
    (8, 2, 150, 260, 128, 1, 1),      # the vector layout but for the bases: 2-byte aligned
    (64, 16, 300, 200, 64, 0, 3),
    (8, 2, 140, 7, 128, 0, 0),        # V^T rows shorter than a piece
    (4, 2, 140, 9, 40, 1, 0),
    (32, 8, 1, 1001, 100, 0, 0),      # decode, split
    (8, 2, 5, 517, 33, 1, 1),         # decode, three row blocks
    (64, 64, 1, 2309, 128, 0, 5),     # decode, V^T groups of four steps and a one-key tail
    (4, 2, 3, 5, 128, 1, 0),          # decode, V^T rows shorter than a piece
    (4, 2, 2, 40, 5, 0, 0),
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_unaligned(oracle, case):
    Hq, Hkv, Sq, Sk, D, causal, off = case
    print("case", case, flush=True)
    Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 991 + D)
    Vt = np.ascontiguousarray(V.reshape(Hkv, Sk, D).transpose(0, 2, 1)).ravel()
    rows = oracle.ref_rowset(Sq, 16)
    R = oracle.attn_ref(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, rows, nthreads=8)
    for vt in (0, 1):
        O = attend(Q, K, Vt if vt else V, Hq, Hkv, Sq, Sk, D, causal, vt, off)
        # the reference's pass rule; P rounded to bf16 (2^-9 of a weight) stays well below it
        ok, mad, maxref, nbad = oracle.cmp_rows(R, O, Hq, Sq, D, rows)
        print("   vt=%d err/scale=%.2e nbad=%d" % (vt, mad / maxref, nbad), flush=True)
        assert ok and nbad == 0, (case, vt, mad, maxref)


@pytest.mark.parametrize("Hkv,Sk,D", [(3, 129, 65), (2, 1, 300), (1, 260, 7), (2, 135, 64),
                                      (1, 7, 128), (5, 128, 70)])
def test_unaligned_pack(Hkv, Sk, D):
    V = np.arange(Hkv * Sk * D, dtype=np.uint32).astype(np.uint16)
    src, addr = guarded(V, 1)
    dst, out = guarded(np.zeros(V.size, np.uint16), 3)
    ts.pack_v_full(addr, out, Hkv, Sk, D)
    ts.synchronize()
    raw = dst.download(np.uint16)
    got = raw[PAD + 3:PAD + 3 + V.size].reshape(Hkv, D, Sk)
    assert np.array_equal(got, V.reshape(Hkv, Sk, D).transpose(0, 2, 1))
    assert np.all(raw[:PAD + 3] == 0xFFFF) and np.all(raw[PAD + 3 + V.size:] == 0xFFFF)
    src.free()
    dst.free()


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, causal: 192-wide tiles (D in (128, 192]) and the last of the 256-wide
    (8, 2, 300, 640, 136, 0), (8, 2, 300, 640, 192, 1), (8, 2, 300, 640, 200, 1),
    (6, 3, 129, 65, 160, 0), (16, 4, 40, 129, 184, 1),
    # 8 waves: tiles of 32 keys (D > 192) and 64, whole and ragged, one to many of them
    (48, 8, 700, 200, 256, 0), (160, 16, 700, 700, 200, 1), (72, 8, 400, 832, 256, 1),
    (48, 8, 700, 24, 256, 0), (256, 32, 256, 40, 208, 0), (48, 8, 700, 328, 136, 0),
    (160, 16, 641, 648, 192, 1), (256, 32, 256, 64, 192, 0),
    # and without the vector layout
    (4, 2, 257, 333, 189, 0), (4, 2, 300, 301, 250, 1), (2, 1, 129, 5, 201, 0), (3, 1, 500, 77, 131, 1),
    (256, 16, 500, 507, 256, 1),
])
def test_wide_head_dims(oracle, case):
    """The wide tiles' loop without a rescale, and its way out: keys whose scores jump from tile to
    tile (up to 2^9 against a stale maximum of the row) fail the sum test in the middle of it."""
    Hq, Hkv, Sq, Sk, D, causal = case
    print("case", case, flush=True)
    Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 4242 + D)
    K = K.reshape(Hkv, Sk, D).copy()
    K[:, 70::97] = (oracle.f32_to_bf16((oracle.bf16_to_f32(K[:, 70::97].ravel()) * 16))).reshape(
        K[:, 70::97].shape)
    rows = oracle.ref_rowset(Sq, 16)
    R = oracle.attn_ref(Q, K.ravel(), V, Hq, Hkv, Sq, Sk, D, causal, rows, nthreads=8)
    for vt in (0, 1):
        Vin = np.ascontiguousarray(V.reshape(Hkv, Sk, D).transpose(0, 2, 1)).ravel() if vt else V
        if Hq >= 48 or D % 8:  # the 8-wave cases
            kt = 64 if D <= 192 and D % 8 == 0 and not (vt and Sk % 8) else 32
            name = ts.attn_flash_plan(Hq, Hkv, Sq, Sk, D, causal, v_prepacked=vt)[0][0]
            assert "<%d, %d, 8, " % (192 if D <= 192 else 256, kt) in name, (case, vt, name)
        O = attend(Q, K.ravel(), Vin, Hq, Hkv, Sq, Sk, D, causal, vt, 0)
        ok, mad, maxref, nbad = oracle.cmp_rows(R, O, Hq, Sq, D, rows)
        print("   vt=%d err/scale=%.2e nbad=%d" % (vt, mad / maxref, nbad), flush=True)
        assert ok and nbad == 0, (case, vt, mad, maxref)


TWO_BLOCKS = {(256, 32, 8, 2053, 128, 1), (192, 64, 12, 1000, 96, 1), (192, 64, 12, 1001, 97, 0),
              (128, 2, 1, 32700, 40, 0), (64, 16, 16, 5000, 64, 1)}


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, causal: three and four 16-row blocks per kv head, one per workgroup
    (256, 32, 8, 517, 128, 1),   # four blocks, a five-key last tile
    (192, 64, 12, 400, 96, 1),   # three blocks, the last of 4 rows
    (192, 64, 12, 401, 97, 0),   # unaligned
    (64, 1, 1, 16500, 40, 0),    # one kv head: 65 splits
    (64, 16, 16, 1024, 64, 1),
    # and two per workgroup (TWO_BLOCKS)
    (256, 32, 8, 2053, 128, 1), (192, 64, 12, 1000, 96, 1), (192, 64, 12, 1001, 97, 0),
    (128, 2, 1, 32700, 40, 0),   # the cap of 64 splits
    (64, 16, 16, 5000, 64, 1),
    # merges: splits of 3 to 64, column counts that end inside a 4-float piece
    (2, 2, 1, 300, 7, 0), (5, 1, 1, 1500, 101, 0), (8, 8, 1, 4100, 256, 0), (1, 1, 1, 8192, 250, 0),
    (3, 1, 4, 1030, 66, 1), (512, 128, 4, 1000, 128, 1),
])
def test_decode_groups_and_merges(oracle, case):
    Hq, Hkv, Sq, Sk, D, causal = case
    plans = [ts.attn_flash_plan(Hq, Hkv, Sq, Sk, D, causal, v_prepacked=vt) for vt in (0, 1)]
    print("case", case, plans, flush=True)
    if ts.device_info()["cus"] == 256:
        for p in plans:
            assert (", 2 blocks" in p[0][0]) == (case in TWO_BLOCKS), p
    Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 777 + D)
    Vt = np.ascontiguousarray(V.reshape(Hkv, Sk, D).transpose(0, 2, 1)).ravel()
    rows = oracle.ref_rowset(Sq, 16)
    R = oracle.attn_ref(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, rows, nthreads=8)
    O = attend(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, 0, 0)
    ok, mad, maxref, nbad = oracle.cmp_rows(R, O, Hq, Sq, D, rows)
    print("   err/scale=%.2e nbad=%d" % (mad / maxref, nbad), flush=True)
    assert ok and nbad == 0, (case, mad, maxref)
    # the same order of sums from V^T, whichever kernel reads it
    assert np.array_equal(O, attend(Q, K, Vt, Hq, Hkv, Sq, Sk, D, causal, 1, 0)), case


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, causal, base offset in elements, what the plan's first kernel holds for
    # row-major V and for V^T: rows shorter than a piece (", short": of Q, K and V, or of V^T)
    (4, 2, 1, 300, 1, 0, 0, ", short", ", short"),
    (4, 2, 2, 5, 1, 1, 0, ", short", ", short"),
    (4, 2, 1, 3, 2, 0, 1, ", short", ", short"),
    (8, 2, 3, 777, 7, 1, 0, ", short", ", short"),
    (64, 64, 1, 2309, 7, 0, 3, ", short", ", short"),
    (256, 4, 1, 16500, 5, 0, 0, ", short, 2 blocks", ", short, 2 blocks"),
    (4, 2, 1, 7, 100, 0, 0, "<128, ", ", short"),
    (4, 2, 2, 7, 200, 1, 0, "<256, ", ", short"),
    # the staged V^T kernel's limits: D > 32, more than two 128-key steps per part
    (512, 256, 1, 700, 32, 0, 1, "attn_decode_kernel<64", "attn_decode_kernel<64"),
    (512, 256, 1, 700, 33, 0, 0, "attn_decode_kernel<64", "attn_decode_vt_kernel<64"),
    (512, 256, 1, 510, 33, 0, 0, "attn_decode_kernel<64", "attn_decode_kernel<64"),
    (1024, 512, 1, 257, 121, 0, 0, "attn_decode_kernel<128", "attn_decode_vt_kernel<128"),
    # pieces at a row's end in both tensors, D % 8 of every kind, at each tile width
    (8, 2, 1, 1001, 9, 0, 0, "<64, ", "<64, "), (8, 2, 1, 1001, 63, 0, 0, "<64, ", "<64, "),
    (8, 2, 5, 133, 65, 1, 0, "<128, ", "<128, "), (8, 2, 1, 1023, 127, 0, 1, "<128, ", "<128, "),
    (8, 2, 1, 1023, 129, 0, 0, "<256, ", "<256, "), (8, 2, 9, 141, 255, 1, 0, "<256, ", "<256, "),
    (64, 64, 1, 2309, 250, 0, 0, "<256, ", "<256, "), (8, 2, 1, 1000, 256, 0, 1, "<256, ", "<256, "),
    (8, 2, 1, 1000, 104, 0, 1, "<128, ", "<128, "),
])
def test_unaligned_decode(oracle, case):
    """Decode kernels on tensors without the vector layout, at both sides of the rules between them.
    Infinite values beyond what a row may see must not reach it: the last key's K row holds some
    where the causal mask hides it from the first rows."""
    Hq, Hkv, Sq, Sk, D, causal, off, want, want_t = case
    print("case", case, flush=True)
    if ts.device_info()["cus"] == 256 and off == 0:
        for vt, w in ((0, want), (1, want_t)):
            name = ts.attn_flash_plan(Hq, Hkv, Sq, Sk, D, causal, v_prepacked=vt)[0][0]
            if D % 8 or (vt and Sk % 8):
                assert w in name, (case, vt, name)
    Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 313 + D)
    hide = causal and Sq > 1
    if hide:
        K = K.reshape(Hkv, Sk, D).copy()
        K[:, -1, ::3] = 0x7F80  # only the last query row of a head sees it: not compared
        K = K.ravel()
    Vt = np.ascontiguousarray(V.reshape(Hkv, Sk, D).transpose(0, 2, 1)).ravel()
    rows = np.arange(Sq - 1 if hide else Sq, dtype=np.int32)
    R = oracle.attn_ref(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, rows, nthreads=8)
    for vt in (0, 1):
        O = attend(Q, K, Vt if vt else V, Hq, Hkv, Sq, Sk, D, causal, vt, off)
        ok, mad, maxref, nbad = oracle.cmp_rows(R, O, Hq, Sq, D, rows)
        print("   vt=%d err/scale=%.2e nbad=%d" % (vt, mad / maxref, nbad), flush=True)
        assert ok and nbad == 0, (case, vt, mad, maxref)


@pytest.mark.parametrize("case", [
    # Hq, Hkv, Sq, Sk, D, causal, base offset: prefill of rows shorter than a piece
    (2, 1, 100, 1, 1, 0, 0), (2, 1, 100, 7, 1, 1, 0), (2, 1, 100, 8, 1, 0, 1),  # heads of 1-8 elements
    (2, 2, 70, 2, 3, 0, 0), (2, 2, 70, 3, 3, 1, 1), (2, 1, 70, 1, 7, 0, 0), (2, 1, 70, 2, 5, 1, 0),
    (3, 3, 130, 129, 1, 0, 0), (3, 3, 130, 130, 3, 1, 0), (3, 3, 130, 257, 7, 0, 3),  # short last tiles
    (4, 2, 200, 128, 5, 0, 0), (4, 2, 200, 263, 2, 1, 1), (64, 64, 65, 385, 6, 1, 0),
    (8, 4, 101, 1801, 7, 0, 0), (8, 4, 300, 900, 3, 1, 0),  # key splits
    (32, 8, 20, 333, 4, 1, 1), (600, 600, 140, 300, 5, 0, 0),
])
def test_short_row_prefill(oracle, case):
    Hq, Hkv, Sq, Sk, D, causal, off = case
    print("case", case, flush=True)
    Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 17 + D)
    Vt = np.ascontiguousarray(V.reshape(Hkv, Sk, D).transpose(0, 2, 1)).ravel()
    rows = oracle.ref_rowset(Sq, 16)
    R = oracle.attn_ref(Q, K, V, Hq, Hkv, Sq, Sk, D, causal, rows, nthreads=8)
    for vt in (0, 1):
        O = attend(Q, K, Vt if vt else V, Hq, Hkv, Sq, Sk, D, causal, vt, off)
        ok, mad, maxref, nbad = oracle.cmp_rows(R, O, Hq, Sq, D, rows)
        print("   vt=%d err/scale=%.2e nbad=%d" % (vt, mad / maxref, nbad), flush=True)
        assert ok and nbad == 0, (case, vt, mad, maxref)
