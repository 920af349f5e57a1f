"""int4_plan (int4_gemm_plan.hpp, built here for the host): what it hands to the launcher exists, covers the product and stays within the
scratch that callers have."""
import ctypes as C
import os
import random
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "int4_gemm_plan.hpp"
extern "C" void plan(size_t m, size_t n, size_t kt, int gm, int zp, long *out) {
  const yscv::RingPlan p = yscv::int4_plan(m, n, kt, 256, gm, zp != 0);
  out[0] = p.one, out[1] = p.second, out[2] = (long)p.split_col, out[3] = p.splits, out[4] = p.kt_per;
}
"""


def test_plans_cover_the_product(tmp_path):
    (tmp_path / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "yscv_amd", "csrc"), str(tmp_path / "plan.cpp"), "-o",
                    str(tmp_path / "plan.so")], check=True)
    lib = C.CDLL(str(tmp_path / "plan.so"))
    lib.plan.argtypes = [C.c_size_t] * 3 + [C.c_int] * 2 + [C.c_void_p]
    rng, out, kinds = random.Random(1), (C.c_long * 5)(), set()
    for _ in range(20000):
        m, n, kt = rng.randint(17, 2300), int(64 * 2000 ** rng.random()), rng.randint(1, 128)
        lib.plan(m, n, kt, rng.randint(0, 2), rng.randint(0, 1), out)
        one, second, col, splits, per = out
        kinds.add((one, splits > 1, second >= 0))
        assert (0 <= one < 5 or 16 <= one < 20) and (second < 5 or 16 <= second < 20), (m, n, kt)  # shapes the launcher has
        assert m > 64 or one < 5
        assert second < 0 or (0 < col < n and col % 16 == 0 and splits == 1), (m, n, kt)
        assert splits >= 1 and splits * per >= kt > (splits - 1) * per, (m, n, kt)
        assert splits == 1 or splits * m * n * 4 + m * kt * 256 <= 31 << 20, (m, n, kt)
    assert {(16, False, False), (18, True, False), (19, True, False), (16, False, True)} <= kinds
