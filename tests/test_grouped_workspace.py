"""Workspace of the grouped GEMM: a call asks for the areas that it can use and for no other (host arithmetic, no GPU)."""
import os

import pytest

from flaggems_amd import _lib

BASE = _lib.FG_WORKSPACE_COUNTER_BYTES + (64 << 20)  # counters and partial sums of cut tiles


def _up(n):
    return -(-n // 256) * 256


def _sorted(M, N, K):
    return _lib.load().fg_grouped_block_fp8_gemm_workspace_bytes(M, N, K)


def _gathered(M, N, K, a_rows, groups):
    return _lib.load().fg_grouped_block_fp8_gemm_gathered_workspace_bytes(M, N, K, a_rows, groups)


@pytest.fixture(autouse=True)
def _built():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("shared library not built on this host")


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (1023, 4096, 14336), (1024, 4096, 14336), (8192, 4096, 14336), (65536, 4096, 14336)])
def test_rows_in_sorted_order_ask_for_no_copy(M, N, K):
    """The second product of an expert layer (Mixtral on 4096 tokens: M = 8192, K = 14336) and callers without an index."""
    assert _sorted(M, N, K) == BASE + _up(4 * M * (K // 128)) + 16 * (M + 1)


@pytest.mark.parametrize("M,N,K,a_rows,groups,copied", [
    (8192, 28672, 4096, 4096, 8, True),      # Mixtral's gate/up product on 4096 tokens
    (1040, 16640, 256, 4096, 5, True),       # more source rows than sorted ones
    (1040, 16640, 256, 300, 5, True),
    (1040, 8448, 256, 4096, 5, False),       # one round of tiles
    (500, 28672, 4096, 512, 2, True),        # few rows, many tiles
    (1024, 28672, 4096, 512, 16, False),     # 64 rows a group: 128-row tiles read through the index
    (300, 28672, 4096, 150, 8, False),       # streaming kernel
    (2048, 512, 4096, 1024, 4, False),
    (300000, 28672, 4096, 150000, 8, False),  # over 1 GiB
])
def test_gathered_rows(M, N, K, a_rows, groups, copied):
    KB = K // 128
    want = (_up(4 * M * KB) + _up(M * K)) if copied else _up(4 * a_rows * KB)
    assert _gathered(M, N, K, a_rows, groups) == BASE + 16 * (M + 1) + want


def test_no_workspace_for_what_is_refused():
    assert _sorted(0, 128, 128) == 0 and _sorted(16, 128, 100) == 0
    assert _gathered(0, 128, 128, 4, 2) == 0 and _gathered(16, 128, 100, 4, 2) == 0 and _gathered(16, 128, 128, 0, 2) == 0
