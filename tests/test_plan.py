"""How the prefill kernels share their work out (mxh_plan.h, host code): every
plan covers K and the keys, keeps within the scratch it is given, and follows
the device's CU count (a partitioned GPU shows 32, 64 or 128).
"""
from __future__ import annotations

import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

HDR = Path(__file__).resolve().parent.parent / "minxfmr.cpp_amd" / "csrc" / "hip"
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
SRC = """
#include "mxh_plan.h"
using namespace mxh;
extern "C" void gemm(int f, int m, int n, int k, int cus, size_t bytes, int* o) {
    const GemmPlan p = gemm_plan((GemmFmt)f, m, n, k, cus, bytes);
    o[0] = p.tile, o[1] = p.blocks, o[2] = p.splits;
}
extern "C" void attn(int hd, int64_t wgs, int stages, size_t wg_bytes, int cus, size_t bytes, int* o) {
    const AttnPlan p = attention_plan(hd, wgs, stages, wg_bytes, cus, bytes);
    o[0] = p.stages, o[1] = p.splits;
}
"""
MIB = 1 << 20


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{HDR}", str(d / "plan.cpp"), "-o",
                    str(d / "plan.so")], check=True)
    return C.CDLL(str(d / "plan.so"))


def gemm(lib, f, m, n, k, cus, scratch=64 * MIB):
    o = (C.c_int * 3)()
    lib.gemm(f, m, n, k, cus, C.c_size_t(scratch), o)
    return tuple(o)


def attn(lib, hd, wgs, stages, cus, scratch=64 * MIB):
    o = (C.c_int * 2)()
    lib.attn(hd, C.c_int64(wgs), stages, C.c_size_t(64 * (hd + 2) * 4), cus, C.c_size_t(scratch), o)
    return tuple(o)


@pytest.mark.parametrize("cus", [32, 64, 128, 256])
def test_plans_cover_the_work(lib, cus):
    for f in range(8):
        for m in (1, 31, 129, 512):
            for n in (1, 300, 4096, 151936):
                for k in (256, 2304, 4096, 16384):
                    for scratch in (0, MIB, 64 * MIB):
                        tile, blocks, splits = gemm(lib, f, m, n, k, cus, scratch)
                        assert 0 <= tile < 4 and (f != 7 or tile != 0)  # (no 128 x 256 tile for Q6_K)
                        assert (splits - 1) * blocks < k // 256 <= splits * blocks
                        assert splits == 1 or 4 * splits * m * n <= scratch
    for hd in (32, 64, 128):
        for wgs in (1, 8, 64, 4096):
            for stages in (1, 7, 128, 5000):
                for scratch in (0, MIB, 64 * MIB):
                    per, splits = attn(lib, hd, wgs, stages, cus, scratch)
                    assert (splits - 1) * per < stages <= splits * per
                    assert splits == 1 or wgs * splits * 64 * (hd + 2) * 4 <= scratch


def test_plans_follow_the_cu_count(lib):
    # 64 weight tiles: a quarter of 256 CUs, so K is split; twice a 32-CU partition, so it is not
    assert gemm(lib, 1, 32, 16384, 8192, 256)[2] >= 2
    assert gemm(lib, 1, 32, 16384, 8192, 32)[2] == 1
    # 8 workgroups over 121 stages
    wide, narrow = attn(lib, 128, 8, 121, 256)[1], attn(lib, 128, 8, 121, 32)[1]
    assert wide > 2 * narrow >= 2


def test_both_orders_of_a_type_have_one_plan(lib):
    # (GGUF order, tiled) of Q4_K, Q5_K, Q8_0: the same K split, so the same bits
    for gguf, tiled in ((0, 1), (2, 3), (4, 5)):
        for m in (1, 19, 64, 200, 512):
            for n in (256, 1030, 4096, 28672):
                for k in (256, 512, 4096, 14336):
                    assert gemm(lib, gguf, m, n, k, 256) == gemm(lib, tiled, m, n, k, 256)
