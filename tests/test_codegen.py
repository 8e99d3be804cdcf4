"""CPU checks of the generated gfx950 code of this repository's own build (no GPU needed).

The LDS-DMA kernels (the fast prefill and the V^T decode) order their DMA and their LDS reads
themselves: each wave waits for its own DMA (vmcnt(0)) right before the barrier that ends a tile.
The compiler can also add vmcnt waits on the DMA in flight before LDS reads inside the key loop
(it does so for a kernel that makes no out-of-line call, since it cannot tell the two tile
buffers apart), which serialises each tile with the next tile's load: 3-15% slower on the
prefill shapes. This test reads the disassembly of the built library and fails if any such
wait appears after a kernel's first MFMA.
"""
import os
import re
import shutil
import subprocess
import tempfile

import pytest

from transfer_station_amd import build as _build

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
OBJDUMP = os.path.join(ROCM, "llvm", "bin", "llvm-objdump")


@pytest.fixture(scope="module")
def funcs(tmp_path_factory):
    """Instruction lists by function name of the built library's gfx950 code object."""
    tmp_path = tmp_path_factory.mktemp("codegen")
    lib = _build.lib_path()
    if not os.path.exists(lib):
        pytest.skip("library not built")
    if not os.access(OBJDUMP, os.X_OK):
        pytest.skip("llvm-objdump not found under %s" % ROCM)
    # --offloading writes the bundled code objects next to its input: work on a copy.
    copy = os.path.join(str(tmp_path), "lib.so")
    shutil.copy(lib, copy)
    subprocess.run([OBJDUMP, "--offloading", copy], cwd=str(tmp_path), check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    objs = [f for f in os.listdir(str(tmp_path)) if f.endswith("gfx950")]
    assert len(objs) == 1, os.listdir(str(tmp_path))
    out = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", os.path.join(str(tmp_path), objs[0])],
                         check=True, stdout=subprocess.PIPE, universal_newlines=True).stdout
    funcs, cur = {}, None
    for line in out.split("\n"):
        m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if m:
            cur = funcs.setdefault(m.group(1), [])
            continue
        if cur is not None and line.startswith("\t"):
            ins = line.strip().split("//")[0].strip()
            if ins:
                cur.append(ins)
    return funcs


def test_lds_dma_kernels_have_no_compiler_dma_waits(funcs):
    kernels = {n: ins for n, ins in funcs.items()
               if "attn_prefill_fast_kernel" in n or "attn_decode_vt_kernel" in n}
    assert len(kernels) >= 40, sorted(funcs)[:5]
    bad = {}
    for name, ins in kernels.items():
        first = next((i for i, x in enumerate(ins) if x.startswith("v_mfma")), None)
        assert first is not None, name
        for i in range(first, len(ins)):
            if ins[i].startswith("s_waitcnt") and "vmcnt" in ins[i]:
                nxt = [y for y in ins[i + 1:i + 6] if not y.startswith(("s_waitcnt", "s_nop"))]
                if nxt and nxt[0].startswith("ds_read"):
                    bad.setdefault(name, []).append(i)
    assert not bad, "vmcnt waits before LDS reads in the key loop of %d kernels, e.g. %s" % (
        len(bad), sorted(bad)[0])


def test_kernels_make_only_the_deliberate_library_call(funcs):
    """HIP's id builtins are out-of-line calls in this build; the kernels read the ids directly,
    except one threadIdx.x in each LDS-DMA kernel (the call that keeps the loop above free of
    compiler DMA waits): the fast and persistent prefills and the V^T decode."""
    for name, ins in funcs.items():
        if not name.startswith("_Z") or "attn_" not in name:
            continue
        calls = sum(1 for x in ins if x.startswith("s_swappc"))
        want = 1 if any(k in name for k in ("attn_prefill_fast_kernel", "attn_prefill_persist_kernel",
                                            "attn_decode_vt_kernel")) else 0
        assert calls == want, (name, calls)


def test_split_merge_loads_are_in_flight_together(funcs):
    """The merge of up to 64 partials is a chain of latencies: its NL column loads per thread are
    issued back to back, with no wait and no branch between them (branches around the loads cost
    short merges 1-2 us)."""
    kernels = {n: ins for n, ins in funcs.items() if "attn_mergew_kernel" in n}
    assert kernels
    for name, ins in kernels.items():
        want = int(re.search(r"attn_mergew_kernelILi(\d+)E", name).group(1))
        best = run = 0
        for x in ins:
            if x.startswith(("s_waitcnt", "s_cbranch", "s_branch", "s_barrier")):
                run = 0
            elif x.startswith("global_load_dwordx4"):
                run += 1
                best = max(best, run)
        assert best >= want, (name, best, want)


def _decode_kernels(funcs, al):
    """(DP, V^T, instructions) of the decode kernels of one alignment class (0: unaligned)."""
    out = []
    for n, ins in funcs.items():
        m = re.search(r"attn_decode_kernelILi(\d+)ELb(\d)EL[ib](\d)ELb(\d)E", n)
        if m and int(m.group(3)) == al:
            out.append((n, int(m.group(1)), int(m.group(4)), ins))
    return out


def test_unaligned_decode_loads_are_in_flight_together(funcs):
    """Unaligned rows are read in two steps, so that a tile's K pieces are all in flight before the
    first is waited for and shifted into place (a shift at the load made decode at small head
    dims one memory latency per piece)."""
    kernels = _decode_kernels(funcs, 0)
    assert kernels
    for name, dp, vt, ins in kernels:
        best = run = 0
        for x in ins:
            if x.startswith("s_waitcnt") and "vmcnt" in x:
                run = 0
            elif x.startswith("global_load_dwordx4"):
                run += 1
                best = max(best, run)
        assert best >= dp // 16, (name, best)  # 2 x DP / 32 K pieces


def test_decode_kernels_do_not_spill():
    """attn_decode_kernel asks for two waves per SIMD, which leaves 256 registers: no instance may
    pay for that with spills on every tile (unaligned rows past D = 128 once spilled 90-112, up to
    1.8 times the time without)."""
    readelf = os.path.join(ROCM, "llvm", "bin", "llvm-readelf")
    if not os.path.exists(_build.lib_path()):
        pytest.skip("library not built")
    if not os.access(readelf, os.X_OK) or not os.access(OBJDUMP, os.X_OK):
        pytest.skip("llvm tools not found under %s" % ROCM)
    with tempfile.TemporaryDirectory() as tmp:
        copy = os.path.join(tmp, "lib.so")
        shutil.copy(_build.lib_path(), copy)
        subprocess.run([OBJDUMP, "--offloading", copy], cwd=tmp, check=True,
                       stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        obj = [f for f in os.listdir(tmp) if f.endswith("gfx950")]
        assert len(obj) == 1, obj
        notes = subprocess.run([readelf, "--notes", os.path.join(tmp, obj[0])], check=True,
                               stdout=subprocess.PIPE, universal_newlines=True).stdout
    spills = {m.group(1): int(m.group(2)) for m in re.finditer(
        r"\.symbol: +'?(\S*?attn_decode_kernel\S*?)\.kd'?\n(?:.*\n)*? +\.vgpr_spill_count: +(\d+)",
        notes)}
    assert len(spills) >= 40, len(spills)
    bad = {n: c for n, c in spills.items() if c}
    assert not bad, bad


def test_short_row_prefill_loads_rows_whole(funcs):
    """Head dims below 8: a K or V row is one 16-byte load (element by element, in a loop that waited
    for each, these prefills took up to 1.5 times as long)."""
    kernels = {n: ins for n, ins in funcs.items()
               if re.search(r"attn_prefill_fast_kernelILi64ELi128ELi4E.*Li2EE", n)}
    assert len(kernels) == 4, sorted(kernels)
    for name, ins in kernels.items():
        # K, and V or V^T: four pieces per thread each, at the first tile and in the loop
        assert sum(x.startswith("global_load_dwordx4") for x in ins) >= 16, name
