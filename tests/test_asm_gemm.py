"""tile_gemm issues its weight loads and LDS reads as inline asm, which the compiler does not know to be in flight.
Compiles verify_sampler.hip (hipcc, no GPU) and checks every instantiation's gfx950 code: no destination register
of a weight load (global_load_dwordx4) or an LDS read (ds_read_b128) is read, copied or reused on any path before a
wait that covers the load, no MFMA's result is read before it is there, and nothing is spilled (a spill could store
a register whose load has not landed)."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "nano-vllm-spec-decode_amd")
sys.path.insert(0, PKG)
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

from asm_paths import early_mfma_reads, function_lines, unsafe_in_flight  # noqa: E402


@pytest.fixture(scope="module")
def device_asm(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    import build_ext
    out = str(tmp_path_factory.mktemp("asm") / "vs.s")
    cmd = [hipcc, *build_ext.DEVICE, *build_ext.COMMON, "--cuda-device-only", "-S",
           os.path.join(build_ext.CSRC, "verify_sampler.hip"), "-o", out]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-3000:]
    return open(out).read()


def _kernels(asm):
    return sorted(set(re.findall(r"^(_ZN2sd6lmhead9tile_gemm\w+):", asm, re.M)))


def test_tile_gemm_loads_complete_before_use(device_asm):
    symbols = _kernels(device_asm)
    assert len(symbols) == 11, symbols     # one per workgroup shape
    for symbol in symbols:
        bad, loads, reads = unsafe_in_flight(function_lines(device_asm, symbol))
        tn, tm, da = (int(x) for x in re.search(r"TileILi(\d+)ELi(\d+)ELi\d+ELi\d+ELi(\d+)E", symbol).groups())
        # the first DA - 1 steps' loads and one step's reads, then both for each of the DA steps of the loop
        assert loads >= tn * (2 * da - 1) and reads >= tm * (da + 1), (symbol, loads, reads)
        assert not bad, (symbol, bad[:4])
        scratch = re.search(r"; ScratchSize: (\d+)", device_asm[device_asm.index("\n" + symbol + ":"):])
        assert scratch and int(scratch.group(1)) == 0, symbol


def test_tile_gemm_waits_for_its_mfmas(device_asm):
    """The MFMAs are inline asm too: nothing but an MFMA touches a result before it is there (the sums between two
    ranges and the epilogue wait by s_nop), in every instantiation. Without those waits the check finds reads too early
    in the shape that has the fewest instructions between."""
    found = 0
    for symbol in _kernels(device_asm):
        lines = function_lines(device_asm, symbol)
        bad = early_mfma_reads(lines)
        assert not bad, (symbol, bad[:4])
        found += len(early_mfma_reads([(t, a) for t, a in lines if t != "s_nop 15"]))
    assert found


def test_check_finds_a_wait_too_short(device_asm):
    """The check itself: each counted wait of a kernel's loop lengthened by one lets a load through."""
    symbol = _kernels(device_asm)[0]
    lines = function_lines(device_asm, symbol)
    found = {"vmcnt": 0, "lgkmcnt": 0}
    for i, (text, in_asm) in enumerate(lines):
        m = re.match(r"s_waitcnt (vmcnt|lgkmcnt)\(([1-9]\d*)\)", text)
        if in_asm and m:
            planted = list(lines)
            planted[i] = (f"s_waitcnt {m.group(1)}({int(m.group(2)) + 1})", True)
            found[m.group(1)] += bool(unsafe_in_flight(planted)[0])
    assert found["vmcnt"] and found["lgkmcnt"], found
