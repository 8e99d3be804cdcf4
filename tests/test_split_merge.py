"""The merge of 3 to 64 split partials (attn_mergew_kernel) at the edges of its layout: rows per 16
lanes or per wave, 4 or 8 loads per thread, one to eight split groups, column counts that end
inside a 4-float piece and head dims below one, row counts that end inside a workgroup. A decode of
few heads splits its keys into one 128-key step per part, so the key count sets the number of
parts; the scratch is NaN outside of what the parts write."""
import numpy as np
import pytest

import transfer_station_amd as ts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu_present():
    assert ts.device_count() >= 1, "no HIP device visible: GPU tests must run on the MI355X box"


@pytest.mark.parametrize("nsplit", [3, 4, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("D", [1, 2, 3, 4, 7, 33, 64, 130, 250])
def test_merge_layouts(oracle, nsplit, D):
    Sk = 128 * nsplit - 5
    for Hq, Hkv, Sq in ((1, 1, 1), (5, 1, 1), (3, 3, 1), (12, 2, 5)):
        if -(-512 // (Hkv * ((Hq // Hkv * Sq + 15) // 16))) < nsplit:
            continue
        case = (Hq, Hkv, Sq, Sk, D)
        plan = ts.attn_flash_plan(Hq, Hkv, Sq, Sk, D, Sq > 1)
        print("case", case, plan, flush=True)
        if ts.device_info()["cus"] == 256:
            assert plan[-1][0] == "attn_mergew_kernel", case
            assert "nsplit=%d" % nsplit in plan[-1][1].split(), case
        Q, K, V = ts.synth_normal_qkv(Hq, Hkv, Sq, Sk, D, 55 + D + nsplit)
        n = Hq * Sq * D
        bufs = [ts.DeviceBuffer.from_array(a) for a in (Q, K, V)]
        with ts.DeviceBuffer(4 * n + 64) as do, \
                ts.DeviceBuffer(ts.attn_flash_scratch_bytes(D, 128)) as ds:
            do.fill_bytes(0xFF)
            ds.fill_bytes(0xFF)
            ts.attn_flash(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, do.ptr, Hq, Hkv, Sq, Sk, D, Sq > 1,
                          128, ds, 0)
            ts.synchronize()
            raw = do.download(np.uint32)
        for b in bufs:
            b.free()
        assert np.all(raw[n:] == 0xFFFFFFFF), case
        rows = oracle.ref_rowset(Sq, 16)
        R = oracle.attn_ref(Q, K, V, Hq, Hkv, Sq, Sk, D, Sq > 1, rows, nthreads=8)
        ok, mad, maxref, nbad = oracle.cmp_rows(R, raw[:n].view(np.float32), Hq, Sq, D, rows)
        print("   err/scale=%.2e nbad=%d" % (mad / maxref, nbad), flush=True)
        assert ok and nbad == 0, (case, mad, maxref)
