"""The forms of the decoder's attention (attention_plan.hpp, built here for the host) follow the number of CUs."""
import ctypes as C
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "attention_plan.hpp"
extern "C" int chunks(int batch, int hq, int hkv, int hd, int cus) { return yscv::attention_in_chunks(batch, hq, hkv, hd, cus); }
extern "C" int tiles(unsigned heads, unsigned queries, unsigned waves_q, int cus) { return yscv::prompt_row_tiles(heads, queries, waves_q, cus); }
"""


def test_forms_follow_the_cus(tmp_path):
    (tmp_path / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "yscv_amd", "csrc"), str(tmp_path / "plan.cpp"), "-o",
                    str(tmp_path / "plan.so")], check=True)
    lib = C.CDLL(str(tmp_path / "plan.so"))
    for cus in (256, 64, 32, 0):
        n = cus or 256
        for batch in range(1, 40):  # 8 kv heads: chunks while there are fewer pairs than a quarter of the CUs
            assert lib.chunks(batch, 32, 8, 128, cus) == (batch * 8 * 4 < n)
            assert not lib.chunks(batch, 40, 8, 128, cus) and not lib.chunks(batch, 32, 8, 64, cus)
        for queries in (64, 65, 129, 700, 2048):
            for heads, waves_q in ((8, 1), (4, 2), (32, 4)):
                wgs = heads * -(-queries // (32 * waves_q))
                assert lib.tiles(heads, queries, waves_q, cus) == (2 if wgs >= n else 1)
