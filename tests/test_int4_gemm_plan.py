"""The plan of the int4 GEMMs (int4_gemm_plan.hpp, built here for the host): what it names is what the launcher has, and nothing
it could have named instead takes less by its own table, on any number of CUs."""
import ctypes as C
import math
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "int4_gemm_plan.hpp"
extern "C" void plan(size_t m, size_t n, size_t kt, size_t cus, long *out) {
  const yscv::GemmPlan p = yscv::int4_plan(m, n, kt, cus);
  out[0] = p.one, out[1] = p.second, out[2] = (long)p.split_col, out[3] = p.splits, out[4] = p.kt_per;
}
extern "C" int tile_time(int i, double *out) {
  if (i >= (int)(sizeof(yscv::kTileTime) / sizeof(yscv::kTileTime[0]))) return 0;
  const yscv::TileTime &t = yscv::kTileTime[i];
  out[0] = t.tile, out[1] = t.bm, out[2] = t.bn, out[3] = t.full_fixed, out[4] = t.full_kt, out[5] = t.fast_fixed, out[6] = t.fast_kt;
  return 1;
}
"""
RING = {0: (128, 128), 1: (32, 128), 2: (64, 128)}  # the tiles of int4_gemm_ring.hip, rows x columns
WIDE = {16: (256, 256), 17: (256, 192), 18: (128, 256), 19: (128, 192)}  # and of int4_gemm_wide.hip


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    at = tmp_path_factory.mktemp("plan")
    (at / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "yscv_amd", "csrc"), str(at / "plan.cpp"), "-o",
                    str(at / "plan.so")], check=True)
    lib = C.CDLL(str(at / "plan.so"))
    lib.plan.argtypes = [C.c_size_t] * 4 + [C.c_void_p]
    lib.tile_time.argtypes = [C.c_int, C.c_void_p]
    out, row, table = (C.c_long * 5)(), (C.c_double * 7)(), {}
    while lib.tile_time(len(table), row):
        table[int(row[0])] = tuple(row)[1:]
    assert {t: v[:2] for t, v in table.items()} == {**WIDE, 0: RING[0], 2: RING[2]}

    def plan(m, n, kt, cus=256):
        lib.plan(m, n, kt, cus, out)
        return tuple(out)

    plan.table = table
    return plan


def _rounds(row, m, cols, parts, kt, cus):
    bm, bn, full_fixed, full_kt, fast_fixed, fast_kt = row
    tiles = math.ceil(m / bm) * math.ceil(cols / bn) * parts
    full, rest = full_fixed + full_kt * kt, tiles % cus
    return tiles // cus * full + (max(full * rest / cus, fast_fixed + fast_kt * kt) if rest else 0)


def _us(table, plan, m, n, kt, cus):
    one, second, col, parts, per = plan
    if second >= 0:
        return _rounds(table[one], m, col, 1, kt, cus) + _rounds(table[second], m, n - col, 1, kt, cus)
    return _rounds(table[one], m, n, parts, per, cus) + (3.2 + parts * m * n * 8 / 5e6 if parts > 1 else 0)


@pytest.mark.parametrize("cus", [256, 304, 128, 32, 1])
def test_the_cheapest_of_the_tiles_that_exist(planner, cus):
    rng, table = random.Random(cus), planner.table
    sizes = [(2048, 28672, 32), (2048, 14336, 32), (257, 1024, 8), (65, 64, 1)]
    sizes += [(rng.randint(65, 2300), int(64 * 2000 ** rng.random()), rng.randint(1, 128)) for _ in range(3000)]
    for m, n, kt in sizes:
        plan = planner(m, n, kt, cus)
        one, second, col, parts, per = plan
        assert one in table and (second in WIDE or second == -1), (m, n, kt)
        us = _us(table, plan, m, n, kt, cus)
        cap = max(0, min(16 << 20, (31 << 20) - m * kt * 256))
        for t, row in table.items():
            tm, tiles = math.ceil(m / row[0]), math.ceil(m / row[0]) * math.ceil(n / row[1])
            assert us <= _us(table, (t, -1, 0, 1, kt), m, n, kt, cus) * (1 + 1e-9), (m, n, kt, t)
            for p in range(2, min(16, kt // 4) + 1):
                per = math.ceil(kt / p)
                if tiles < cus and p * m * n * 4 <= cap and math.ceil(kt / per) == p:
                    assert us <= _us(table, (t, -1, 0, p, per), m, n, kt, cus) * (1 + 1e-9), (m, n, kt, t, p)
            at = int(tiles // cus * cus // tm * row[1])
            if t in WIDE and 0 < at < n:
                for u in WIDE:
                    assert us <= _us(table, (t, u, at, 1, kt), m, n, kt, cus) * (1 + 1e-9), (m, n, kt, t, u)


# tiles and parts with the shortest time measured (fp16 rows), where the next ones are more than 8 % behind
@pytest.mark.parametrize("m,n,k,one,parts", [
    (604, 27898, 512, 19, 1), (339, 27654, 2048, 19, 1), (229, 7268, 11904, 0, 2), (529, 7761, 6592, 19, 1), (2048, 6144, 4096, 17, 1),
    (512, 2183, 9728, 0, 3), (588, 84770, 512, 19, 1), (337, 1421, 12736, 0, 7), (114, 97967, 512, 19, 1), (92, 65550, 896, 19, 1)])
def test_shapes_that_were_timed(planner, m, n, k, one, parts):
    plan = planner(m, n, -(-k // 128))
    assert (plan[0], plan[3]) == (one, parts) and plan[1] == -1
