"""Grouped GEMM on 256-row tiles with rows read through an index: large problems copy the rows into sorted order first
(gather_rows_kernel in csrc/fp8_gemm_pingpong.hip).  Sizes around its edges: rows that do not fill the last 16, one K-block,
an odd number, entries out of range, both layouts of the scales, the table of tile rows and the scan."""
import pytest
import torch

import flag_gems

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
