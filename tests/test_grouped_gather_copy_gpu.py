"""Grouped GEMM on 256-row tiles with rows read through an index: large problems copy the rows into sorted order first
(gather_rows_kernel in csrc/fp8_gemm_pingpong.hip).  Sizes around its edges: rows that do not fill the last 16, one K-block,
an odd number, entries out of range, both layouts of the scales, the table of tile rows and the scan."""
import pytest
import torch

import flag_gems
from flaggems_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(T, M, N, K, E, seed, column_major):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(T, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w = (0.5 * torch.randn(E, N, K, generator=g, device=DEV)).to(torch.float8_e4m3fn)
    xs = torch.rand(T, K // 128, generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(E, -(-N // 128), K // 128, generator=g, device=DEV) * 0.02 + 0.005
    if column_major:
        xs = xs.t().contiguous().t()
    cuts = torch.sort(torch.randint(0, M + 1, (E - 1,), generator=g, device=DEV))[0]
    ends = torch.cat([cuts, torch.tensor([M], device=DEV)]).int()
    return x, w, xs, ws, ends, g


@pytest.mark.parametrize("T,M,N,K,E,top_k,column_major", [
    (550, 1100, 8200, 256, 3, 2, False),     # 12 rows in the last block of the copy, the segments scanned
    (1100, 1100, 8200, 128, 3, 1, True),     # one K-block
    (200, 1205, 8200, 384, 4, 6, False),     # three K-blocks, more than one row of the sixteen from the same token
    (4096, 1040, 8448, 256, 5, 1, False),    # more source rows than sorted ones
    (2048, 4096, 6144, 2048, 24, 2, False),  # table of tile rows
    # the first four read through the index (one round of tiles); the same edges where the rows are copied
    (550, 1100, 16400, 256, 3, 2, False),
    (1100, 1100, 28704, 128, 3, 1, True),
    (200, 1205, 16400, 384, 4, 6, False),
    (4096, 1040, 16640, 256, 5, 1, False),
    (150, 300, 32776, 384, 2, 2, False),     # few rows, many tiles
])
def test_rows_copied_in_sorted_order(T, M, N, K, E, top_k, column_major):
    x, w, xs, ws, ends, g = _problem(T, M, N, K, E, M + N + K, column_major)
    idx = torch.randint(0, T * top_k, (M,), generator=g, device=DEV).int()
    idx[3], idx[M - 1], idx[17] = -1, T * top_k, 2**31 - 1  # forced into the rows of A
    src = (idx.long().clamp(min=0) // top_k).clamp(max=T - 1)
    got = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], row_index=idx, index_divisor=top_k)
    # the same rows handed over in sorted order: the same products in the same order
    same = flag_gems.grouped_w8a8_block_fp8_matmul(x[src].contiguous(), w, xs[src].contiguous(), ws, ends, [128, 128])
    assert torch.equal(got, same)
    begin = 0
    for e, end in enumerate(ends.tolist()):
        if end > begin:
            a = x[src[begin:end]].float() * xs[src[begin:end]].repeat_interleave(128, 1)
            b = w[e].float() * ws[e].repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]
            want, mag = a @ b.t(), a.abs() @ b.abs().t()
            # half a bf16 step, plus the matrix instruction's alignment of 128 products to the largest one
            assert ((got[begin:end].float() - want).abs() <= want.abs() * 2.0 ** -8 + 4e-4 * mag).all()
        begin = end


@pytest.mark.parametrize("T,M,N,K,E,sums", [(4096, 1040, 16640, 256, 5, 0), (2048, 4096, 6144, 2048, 24, 64)])
def test_workspace_of_the_stated_size_is_enough(T, M, N, K, E, sums):
    """Workspace of exactly fg_grouped_block_fp8_gemm_gathered_workspace_bytes: the rows are copied (they lie behind the counters, the
    partial sums, where K is long enough to be cut, and their scales), nothing is written past its end, and the results are those of the public call."""
    x, w, xs, ws, ends, g = _problem(T, M, N, K, E, M + N, False)
    idx = torch.randint(0, T, (M,), generator=g, device=DEV).int()
    lib = _lib.load()
    size = lib.fg_grouped_block_fp8_gemm_gathered_workspace_bytes(M, N, K, T, E)
    work = torch.zeros(size + 4096, dtype=torch.uint8, device=DEV)
    work[size:] = 0xA5
    c = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    status = lib.fg_grouped_block_fp8_gemm(
        x.data_ptr(), K, w.data_ptr(), K, N * K, xs.data_ptr(), xs.stride(0), xs.stride(1), ws.data_ptr(), ws.stride(1), 1, ws.stride(0),
        ends.data_ptr(), E, idx.data_ptr(), 1, T, 0, None, c.data_ptr(), N, _lib.DTYPE_CODE[torch.bfloat16], M, N, K, 128, 128,
        work.data_ptr(), size, _lib.current_stream_ptr(torch.device(DEV)))
    _lib.check(status, "fg_grouped_block_fp8_gemm")
    at = _lib.FG_WORKSPACE_COUNTER_BYTES + (sums << 20) + -(-4 * M * (K // 128) // 256) * 256
    rows = work[at:at + M * K].view(M, K)
    assert torch.equal(rows, x[idx.long()].view(torch.uint8))
    assert (work[size:] == 0xA5).all()
    same = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], row_index=idx)
    last = int(ends[-1])
    assert torch.equal(c[:last], same[:last])


@pytest.mark.parametrize("divisor", [None, 0, 2])
def test_only_gathered_calls_ask_for_the_copy(divisor, monkeypatch):
    M, N, K, E = 1024, 256, 512, 2
    T = M // 2 if divisor == 2 else M
    x, w, xs, ws, ends, g = _problem(T, M, N, K, E, 7, False)
    idx = None if divisor is None else torch.randperm(M, generator=g, device=DEV).int()
    asked = []
    real = _lib.cached_workspace_bytes
    monkeypatch.setattr(_lib, "cached_workspace_bytes", lambda name, *shape: asked.append((name, shape)) or real(name, *shape))
    flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], row_index=idx, index_divisor=1 if divisor is None else divisor,
                                            scatter_rows=None if divisor is None else M)
    if divisor:
        assert asked == [("fg_grouped_block_fp8_gemm_gathered_workspace_bytes", (M, N, K, T, E))]
    else:
        assert asked == [("fg_grouped_block_fp8_gemm_workspace_bytes", (M, N, K))]
