"""The hand-over rules of csrc/fp8_gemm_rules.h and csrc/fp8_gemm_skinny_plan.h against measurements on an MI355X (256 compute units): shapes on both sides of every
line, with the time of either kernel, so that a rule that moves a line has to answer for them.  Host code only."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flaggems_amd", "csrc")
SHIM = """
#include "%s/fp8_gemm_rules.h"
#include "%s/fp8_gemm_skinny_plan.h"
extern "C" int tall(int block, long long M, long long N, long long kb, long long cus) { return fg::tall_tiles_pay(block != 0, M, N, kb, cus); }
extern "C" int stream_rows(long long M, long long N, long long kb, long long groups, long long cus) {
  return fg::grouped_stream_pass_rows(M, N, kb, groups, cus);
}
extern "C" int parts(long long M, long long N, long long K, long long* rows, long long* back) {
  const fg::DecodeParts d = fg::decode_parts(M, N, K);
  *rows = d.rows, *back = d.back;
  return (int)d.parts;
}
extern "C" int copy_rows(long long M, long long N, long long K, long long groups, long long cus) { return fg::gather_copy_pays(M, N, K, groups, cus); }
extern "C" int skinny(int block, long long M, long long N, long long K, long long ldw, int cus, int* plan) {
  const fg::SkinnyPlan p = fg::plan_skinny(M, N, K, ldw, block != 0, cus);
  if (!p.use) return 0;
  plan[0] = fg::kSkinnyShapes[p.cfg].bm, plan[1] = fg::kSkinnyShapes[p.cfg].bn, plan[2] = p.tiles_m, plan[3] = p.splits;
  return 1;
}
""" % (CSRC, CSRC)


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
    so.stream_rows.argtypes = so.copy_rows.argtypes = [ctypes.c_longlong] * 5
    so.skinny.argtypes = [ctypes.c_int] + [ctypes.c_longlong] * 4 + [ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    so.parts.argtypes = [ctypes.c_longlong] * 3 + [ctypes.POINTER(ctypes.c_longlong)] * 2
    return so


def _skinny(rules, block, M, N, K, ldw=None):
    """(rows a tile, weight rows a tile, rows of tiles, parts of K), or None where another kernel takes the problem."""
    plan = (ctypes.c_int * 4)()
    return tuple(plan) if rules.skinny(block, M, N, K, ldw or K, 256, plan) else None


@pytest.mark.parametrize("block", [True, False])
def test_the_shapes_of_the_deep_stage_kernels_tests_reach_every_form_of_it(rules, block):
    import test_skinny_gpu as T

    forms, rows = set(), {}
    for M, N, K in T.BLOCK_SCALES if block else T.ROW_AND_COLUMN_SCALES:
        plan = _skinny(rules, block, M, N, K)
        assert plan is not None, (M, N, K)
        bm, bn, tiles_m, splits = plan
        forms.add((bm, bn, tiles_m > 1, splits > 1, K // 128 % 2))
        if tiles_m == 1:
            rows.setdefault((bm, bn), []).append(M)
    tiles = [(bm, bn) for bm in (16, 32, 64) for bn in (32, 64, 128)] + [(128, 64)]
    for bm, bn in tiles:
        for several in (False, True) if bm >= 64 else (False,):
            for split in (False, True) if block or bm > 16 else (False,):
                for odd in (0, 1):
                    assert (bm, bn, several, split, odd) in forms
        assert min(rows[bm, bn]) == (1 if bm == 16 else bm // 2 + 1) and max(rows[bm, bn]) >= bm - 1
    if block:
        assert {_skinny(rules, True, *shape)[:2] for shape in T._EVERY_TILE} == set(tiles)
        assert all(_skinny(rules, True, *shape)[3] > 1 for shape in T.WITHOUT_WORKSPACE)
        assert sum(_skinny(rules, True, *shape) is not None for shape in T.SCALES_FAR_APART) >= 12
        assert all(_skinny(rules, True, *shape) is None for shape in T.SHORT_K)


# block scales?, M, N, K, bytes from one weight row to the next, us on the deep-stage kernel, us on the kernel that serves the shape otherwise
DEEP = [
    # 32 weight rows a tile: K = 8192 from 13 rows or in a nearly full round; block scales from 9 rows with short K
    (False, 9, 6592, 8192, 8192, 12.9, 11.8), (False, 10, 6464, 8192, 8192, 12.6, 11.7), (False, 11, 6656, 8192, 8192, 12.7, 12.0),
    (False, 10, 7488, 8192, 8192, 13.7, 13.1), (False, 16, 7232, 8192, 8192, 13.6, 14.0), (False, 14, 6976, 8192, 8192, 13.3, 13.7),
    (False, 12, 8192, 8192, 8192, 13.5, 16.6), (False, 7, 6720, 4096, 4096, 7.9, 7.4), (False, 5, 8000, 4096, 4096, 8.8, 8.1),
    (True, 9, 6400, 4480, 4480, 8.3, 8.0),
    # 64: K = 4096, 8192; longer K with block scales from 13 rows
    (False, 7, 15680, 4096, 4096, 13.4, 14.4), (True, 8, 15552, 4096, 4096, 13.0, 15.4), (True, 15, 12352, 2048, 2048, 7.3, 8.3),
    (True, 9, 16128, 14336, 14336, 41.4, 38.9), (True, 11, 12352, 14336, 14336, 34.2, 33.4), (False, 10, 15936, 3584, 3584, 12.7, 12.0),
    (False, 10, 15552, 5120, 5120, 17.0, 16.0), (False, 14, 14464, 1024, 1024, 5.3, 6.1),
    # 128
    (False, 1, 30272, 8192, 8192, 44.6, 41.0), (True, 13, 32128, 4096, 4096, 24.4, 28.8),
    # rows that lie as far apart as another K's, or K's rows further apart
    (False, 3, 16128, 4096, 4224, 13.8, 13.2), (False, 3, 29056, 4096, 4224, 22.8, 20.4), (False, 8, 25472, 4096, 4224, 20.6, 19.2),
    (True, 14, 30976, 4096, 5120, 24.0, 22.8), (True, 12, 30080, 4096, 4224, 23.0, 21.7), (True, 9, 27648, 4096, 4128, 22.4, 33.8),
    (False, 11, 6720, 4096, 8192, 9.2, 8.0), (True, 15, 6272, 4096, 8192, 8.9, 8.4), (True, 14, 13888, 2048, 2176, 7.7, 8.8),
    # many rows, long K, row and column scales
    (False, 117, 5504, 16128, 16128, 35.9, 32.6), (False, 114, 5632, 16384, 16384, 35.5, 32.1), (False, 103, 5824, 16000, 16000, 33.9, 31.5),
    (False, 71, 5504, 14592, 14592, 27.7, 28.6),
]


@pytest.mark.parametrize("block,M,N,K,ldw,deep,other", DEEP)
def test_deep_stage_kernel_where_it_is_the_faster_one(rules, block, M, N, K, ldw, deep, other):
    assert (_skinny(rules, block, M, N, K, ldw) is not None) == (deep < other)


def test_parts_of_the_rows_stay_inside_the_matrix(rules):
    """Every part begins a part's rows after the one before and ends inside the matrix; only the last one is moved back."""
    rows, back = ctypes.c_longlong(), ctypes.c_longlong()
    taken = 0
    for N, K in ((512, 512), (832, 1152), (576, 7168), (1024, 2048), (1536, 7168), (4096, 512), (6144, 8192), (8192, 1024)):
        for M in range(1, 600):
            n = rules.parts(M, N, K, ctypes.byref(rows), ctypes.byref(back))
            if n == 0:
                continue
            taken += 1
            assert 1 <= rows.value <= 16 and 0 <= back.value < rows.value
            assert (n - 1) * rows.value <= M and n * rows.value - back.value == M
    assert taken > 1000


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


# groups, N, K, rows a group, us on the streaming kernel, us on the persistent one (rows spread at random over the groups)
STREAM = [
    (1, 7168, 256, 4, 12.3, 10.1), (2, 7168, 256, 1, 12.7, 10.5), (2, 2048, 256, 48, 16.6, 11.8), (4, 7168, 128, 32, 15.3, 11.4),
    (8, 7168, 128, 48, 16.8, 13.2), (8, 7168, 256, 48, 17.6, 14.9),
    (8, 16384, 256, 1, 13.0, 20.1), (16, 7168, 256, 24, 15.1, 21.5), (16, 2048, 256, 1, 13.4, 15.7), (256, 7168, 256, 12, 119.6, 176.2),
    (2, 7168, 384, 12, 10.9, 11.9), (8, 7168, 512, 24, 13.0, 16.3), (1, 512, 1024, 4, 9.7, 15.7),
    (32, 4096, 14336, 30, 357.3, 393.1), (32, 4096, 14336, 34, 367.9, 336.2), (32, 4096, 14336, 48, 386.0, 338.9),
    (64, 4096, 14336, 48, 775.7, 671.9), (64, 4096, 6400, 30, 338.7, 357.4), (64, 4096, 6400, 40, 347.5, 315.9),
    (26, 4096, 14336, 37, 333.3, 404.5), (16, 12800, 4096, 48, 195.6, 196.6), (8, 28672, 4096, 48, 190.7, 208.9),
    (8, 4096, 14336, 6, 84.2, 112.8), (64, 2048, 4096, 48, 127.9, 140.3), (64, 2816, 2048, 48, 91.1, 96.6),
    (512, 2048, 4096, 32, 912.0, 816.0), (512, 4096, 1024, 24, 480.7, 496.4), (512, 2048, 4096, 1, 468.0, 2348.0),
]


@pytest.mark.parametrize("groups,N,K,rows,stream,other", STREAM)
def test_streaming_where_it_is_faster(rules, groups, N, K, rows, stream, other):
    assert (rules.stream_rows(groups * rows, N, K // 128, groups, 256) != 0) == (stream < other)


def test_streaming_pass_for_skewed_groups(rules):
    """Large matrices take a pass of twice the average group's rows or more, so that a few long groups do not stream them
    several times (8 x [28672, 4096], 64 rows in one group: 71 us at 16 rows a pass, 41 at 32); 16 - 64 rows always."""
    assert [rules.stream_rows(8 * n, 28672, 32, 8, 256) for n in (1, 6, 7, 8, 16, 24, 25, 48, 49)] == [16, 16, 32, 32, 32, 32, 64, 64, 0]
    assert [rules.stream_rows(n, 6400, 32, 1, 256) for n in (1, 5, 16, 17, 24, 25, 48, 49)] == [16, 16, 16, 32, 32, 64, 64, 0]
    assert [rules.stream_rows(64 * n, 2816, 16, 64, 256) for n in (1, 8, 9, 24, 25, 48, 49)] == [16, 16, 32, 32, 64, 64, 0]
    assert [rules.stream_rows(128 * n, 2816, 16, 128, 256) for n in (1, 8, 9, 24, 25)] == [16, 16, 32, 32, 0]


# groups, N, K, rows, us with the gathered rows copied first, us read through the index
COPY = [
    (8, 28672, 4096, 1118, 266.2, 319.5), (8, 28672, 4096, 7825, 918.0, 1201.3), (6, 12800, 4096, 2020, 143.3, 170.5),
    (6, 4096, 1024, 4071, 50.6, 56.7), (8, 4096, 1024, 4203, 51.6, 57.7), (1, 12800, 4096, 2099, 114.0, 131.6),
    (3, 12800, 4096, 782, 71.8, 82.1), (2, 30016, 7296, 322, 127.0, 151.0),
    (8, 7168, 256, 1139, 24.0, 20.9), (6, 5888, 128, 2267, 21.0, 18.1), (16, 1024, 256, 13882, 28.0, 23.6), (1, 7168, 256, 1787, 22.1, 20.0),
    (6, 1408, 128, 8325, 23.2, 19.9), (2, 1536, 128, 13798, 29.6, 27.0), (2, 3456, 128, 8229, 31.3, 29.2), (64, 576, 256, 10833, 27.4, 24.5),
]


@pytest.mark.parametrize("groups,N,K,rows,copied,indexed", COPY)
def test_gathered_rows_are_copied_where_that_is_faster(rules, groups, N, K, rows, copied, indexed):
    assert bool(rules.copy_rows(rows, N, K, groups, 256)) == (copied < indexed)
