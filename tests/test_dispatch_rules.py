"""The hand-over rules of csrc/fp8_gemm_rules.h against measurements on an MI355X (256 compute units): shapes on both sides of every
line, with the time of either kernel, so that a rule that moves a line has to answer for them.  Host code only."""
import ctypes
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flaggems_amd", "csrc", "fp8_gemm_rules.h")
SHIM = """
#include "%s"
extern "C" int tall(int block, long long M, long long N, long long kb, long long cus) { return fg::tall_tiles_pay(block != 0, M, N, kb, cus); }
""" % HEADER


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    folder = tmp_path_factory.mktemp("rules")
    src, lib = str(folder / "rules.cpp"), str(folder / "rules.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", lib, src], check=True)
    so = ctypes.CDLL(lib)
    so.tall.argtypes = [ctypes.c_int] + [ctypes.c_longlong] * 4
    return so


# block scales?, M, N, K, us on the 256 x 128 tiles, us on the kernel that serves the shape otherwise
TALL = [
    (True, 256, 24576, 1536, 22.4, 25.5), (True, 200, 24576, 1536, 21.5, 24.6),  # one tile row, short K
    (True, 312, 10944, 1408, 18.4, 15.9), (True, 315, 10944, 1152, 16.7, 14.3), (True, 280, 10944, 1920, 21.4, 18.6),  # 258 tiles
    (True, 4048, 1088, 1024, 15.6, 14.2),
    (True, 256, 28672, 4096, 47.2, 59.8), (True, 136, 28672, 4096, 42.4, 52.6),
    (True, 512, 10240, 8192, 70.6, 66.2), (True, 244, 20096, 7424, 69.3, 66.0), (True, 717, 6656, 7680, 67.9, 64.9),
    (True, 184, 20224, 7808, 67.1, 89.7), (True, 2641, 1792, 7296, 56.8, 64.8),
    (False, 312, 10944, 1408, 21.0, 16.3), (False, 315, 10944, 1152, 19.7, 15.2), (False, 256, 24576, 1536, 25.8, 25.3),
    (False, 1844, 4032, 1280, 22.4, 21.4), (False, 200, 16832, 2176, 26.7, 24.7),
    (False, 136, 28672, 4096, 40.4, 45.0), (False, 256, 28672, 4096, 46.0, 50.8), (False, 479, 11648, 4096, 38.5, 43.0),
    (False, 512, 10240, 8192, 62.0, 69.7), (False, 142, 32128, 4736, 48.8, 59.1),
]


@pytest.mark.parametrize("block,M,N,K,tall,other", TALL)
def test_tall_tiles_where_they_are_faster(rules, block, M, N, K, tall, other):
    assert bool(rules.tall(block, M, N, K // 128, 256)) == (tall < other)


@pytest.mark.parametrize("block", [True, False])
def test_tall_tiles_only_where_one_round_takes_them(rules, block):
    for cus in (256, 304, 64):
        for M in (1, 64, 128, 129, 255, 256, 257, 384, 385, 512, 513, 4096):
            for N in (1, 128, 129, 1088, 4096, 10944, 16384, 16385, 32768, 65536):
                for kb in (1, 4, 7, 8, 16, 17, 24, 25, 32, 33, 56, 57, 64, 65, 128):
                    if rules.tall(block, M, N, kb, cus):
                        assert M > 128 and 8 <= kb <= 64
                        assert -(-M // 256) * -(-N // 128) <= cus < -(-M // 128) * -(-N // 128)
