"""tile_gemm issues its weight loads and LDS reads as inline asm, which the compiler does not know to be in flight.
Compiles verify_sampler.hip (hipcc, no GPU) and checks every instantiation's gfx950 code: no destination register
of such a load is read, copied or reused on any path before a wait that covers the load, and nothing is spilled
(a spill could store a register whose load has not landed)."""
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

from asm_paths import function_lines, unsafe_asm_loads  # noqa: E402


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


def test_tile_gemm_loads_complete_before_use(device_asm):
    symbols = sorted(set(re.findall(r"^(_ZN2sd6lmhead9tile_gemm\w+):", device_asm, re.M)))
    assert len(symbols) == 10, symbols     # one per workgroup shape
    for symbol in symbols:
        bad, n = unsafe_asm_loads(function_lines(device_asm, symbol))
        assert n >= 15 and not bad, (symbol, n, bad[:4])
        scratch = re.search(r"; ScratchSize: (\d+)", device_asm[device_asm.index("\n" + symbol + ":"):])
        assert scratch and int(scratch.group(1)) == 0, symbol
