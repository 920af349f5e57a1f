"""Requantisation of a NaN that the compiler knows of (no GPU needed: hipcc cross-compiles to assembly): it is 0, as any other NaN's, and the code
stores it.  A cast of it is undefined, and what it reaches is then left out of the program."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "yscv_amd", "csrc")
SOURCE = """
#include "i8_common.hpp"
__global__ void byte_away(int *out) { out[0] = yscv::requant_int<true>(7, __builtin_nanf(""), 3.0f, 3.0f, 200.0f); }
__global__ void byte_even(int *out) { out[0] = yscv::requant_int<false>(7, __builtin_nanf(""), 3.0f, 3.0f, 200.0f); }
__global__ void dequantised(int *out) {
  out[0] = yscv::requant_dequant_bits(7, 1, __builtin_nanf(""), 3.0f, YSCV_HIP_ROUND_HALF_AWAY, -128.0f, 127.0f, 0.5f);
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_the_result_of_a_known_nan_is_stored(tmp_path):
    src, out = tmp_path / "nan.hip", tmp_path / "nan.s"
    src.write_text(SOURCE)
    proc = subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-I", CSRC, "-S", "--cuda-device-only",
                           "-o", str(out), str(src)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    kernels = out.read_text().split("; -- Begin function ")[1:]
    assert len(kernels) == 3
    for code in kernels:
        assert "global_store_dword" in code, code.split()[0]
