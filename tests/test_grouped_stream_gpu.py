"""The weight-streaming grouped GEMM (few rows per group, csrc/fp8_gemm_stream.hip) and the table of tile rows that the
persistent kernel walks when there are many groups, at the sizes where their index arithmetic can go wrong: groups of 0, 1,
16, 17, 32, 33, 64 rows, one K-block, an odd number of K-blocks, N ending inside an item, ranges that cut an item into
several parts, the largest tables."""
import pytest
import torch

import flag_gems
from flaggems_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FP8 = torch.float8_e4m3fn


def _operands(M, N, K, E, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(FP8)
    w = (0.5 * torch.randn(E, N, K, generator=g, device=DEV)).to(FP8)
    xs = torch.rand(M, -(-K // 128), generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(E, -(-N // 128), -(-K // 128), generator=g, device=DEV) * 0.02 + 0.005
    return x, w, xs, ws


def _reference(x, w, xs, ws, counts):
    """fp32 product of the dequantised operands, group by group, and the sums of |a||b| that bound the error."""
    N, K = w.shape[1:]
    xd = x.float() * xs.repeat_interleave(128, 1)[:, :K]
    out, mag, begin = [], [], 0
    for e, n in enumerate(counts):
        if n:
            wd = w[e].float() * ws[e].repeat_interleave(128, 1)[:, :K].repeat_interleave(128, 0)[:N]
            out.append(xd[begin:begin + n] @ wd.t())
            mag.append(xd[begin:begin + n].abs() @ wd.abs().t())
        begin += n
    return torch.cat(out), torch.cat(mag)


def _close(got, want, mag):
    # half a bf16 step (2^-9 of the value), plus the matrix instruction's alignment of 128 products to the largest one:
    # below 2e-4 of the sum of |a||b|
    assert ((got.float() - want).abs() <= want.abs() * 2.0 ** -8 + 4e-4 * mag).all()


CASES = [
    ([3, 5], 256, 512),
    ([0, 17, 1, 0], 256, 384),                                   # three K-blocks: the last step holds one
    ([1, 0, 2, 33, 16, 7, 0, 40], 1024, 4096),                   # items cut into parts; 1, 2, 16, 33 rows
    ([5, 0, 70], 264, 128),                                      # one K-block; N ends inside a tile (the persistent kernel's, few groups)
    ([5, 0, 70] + [1, 2, 0] * 4, 264, 128),                      # one K-block and more groups: items of one step; N ends inside an item
    ([0, 0, 0, 1], 128, 128),
    ([0] * 9 + [1] + [0] * 3, 128, 128),                         # one step in all
    ([2, 0, 40], 33000, 256),                                    # few groups, but more than one round of tiles
    ([9, 9, 1, 30, 60, 2, 0, 1], 2144, 7168),
    ([48, 64, 32, 16, 65, 1, 0, 47], 512, 1152),                 # 64-row passes, nine K-blocks
    ([i % 5 for i in range(64)], 512, 1024),
    ([1 if i % 3 else 0 for i in range(1024)], 128, 256),        # the largest table of the streaming kernel
    ([i % 2 for i in range(1025)], 128, 256),                    # one group more: the persistent kernel, table of tile rows
    ([60 + i % 9 for i in range(24)], 384, 256),                 # fewest groups with a table; 128-row tiles
    ([130 + 5 * (i % 9) for i in range(40)], 264, 384),          # 256-row tiles
    ([i % 4 for i in range(2048)], 128, 128),                    # the largest table of tile rows
    ([1] * 2049, 128, 128),                                      # beyond it: the groups are scanned
]


@pytest.mark.parametrize("counts,N,K", CASES, ids=lambda v: str(len(v)) if isinstance(v, list) else str(v))
def test_against_fp32(counts, N, K):
    M, E = sum(counts), len(counts)
    x, w, xs, ws = _operands(M, N, K, E, seed=N + K + E)
    ends = torch.tensor(counts).cumsum(0).int().to(DEV)
    got = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128])
    _close(got, *_reference(x, w, xs, ws, counts))
    assert torch.equal(got, flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128]))


@pytest.mark.parametrize("per", [1, 12, 40])
def test_gather_scatter_weights_and_no_workspace(per):
    """Rows through an index with its range check, results scattered and weighted, fp16; the same rows without an index give
    the same bits, and whole items (no workspace) the same values."""
    E, N, K, top_k = 6, 384, 640, 3
    tokens = per * E // top_k + 1
    slots = tokens * top_k
    g = torch.Generator().manual_seed(per)
    expert = torch.randint(0, E, (slots,), generator=g)
    order = torch.argsort(expert, stable=True).int()
    counts = torch.bincount(expert, minlength=E)
    ends = counts.cumsum(0).int().to(DEV)
    x, w, xs, ws = _operands(tokens, N, K, E, seed=per)
    src = (order // top_k).long().to(DEV)
    weight = torch.rand(slots, generator=g).to(DEV) + 0.25
    want, mag = _reference(x[src], w, xs[src], ws, counts.tolist())
    got = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], torch.float16, row_index=order.to(DEV), index_divisor=top_k,
                                                  scatter_rows=slots, row_weights=weight)
    at = order.long().to(DEV)
    _close(got[at], want * weight[at, None], mag * weight[at, None])
    gathered = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], row_index=order.to(DEV), index_divisor=top_k)
    copied = flag_gems.grouped_w8a8_block_fp8_matmul(x[src].contiguous(), w, xs[src].contiguous(), ws, ends, [128, 128])
    assert torch.equal(gathered, copied)
    a, s = x[src].contiguous(), xs[src].contiguous()
    c = torch.empty(slots, N, dtype=torch.bfloat16, device=DEV)
    st = _lib.load().fg_grouped_block_fp8_gemm(
        a.data_ptr(), K, w.data_ptr(), K, N * K, s.data_ptr(), s.stride(0), 1, ws.data_ptr(), ws.stride(1), 1, ws.stride(0),
        ends.data_ptr(), E, None, 1, slots, 0, None, c.data_ptr(), N, _lib.DTYPE_CODE[torch.bfloat16], slots, N, K, 128, 128,
        None, 0, _lib.current_stream_ptr(torch.device(DEV)))
    _lib.check(st, "fg_grouped_block_fp8_gemm")
    _close(c, want, mag)


@pytest.mark.parametrize("per,K", [(2, 640), (14, 1024), (40, 896)])
def test_scale_layouts_and_padded_rows(per, K):
    """Column-major activation scales, and rows of every operand further apart than they are long: the bits of the plain call."""
    E, N = 5, 392
    counts = [per, 0, 2 * per, 1, per]
    M = sum(counts)
    x, w, xs, ws = _operands(M, N, K, E, seed=K)
    ends = torch.tensor(counts).cumsum(0).int().to(DEV)
    base = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128])
    assert torch.equal(flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs.t().contiguous().t(), ws, ends, [128, 128]), base)
    lda, ldb, ldc, rows = K + 48, K + 16, N + 24, N + 3
    xp = torch.full((M, lda), 0x7F, dtype=torch.uint8, device=DEV)  # NaN codes between the rows
    xp[:, :K] = x.view(torch.uint8)
    wp = torch.full((E, rows, ldb), 0x7F, dtype=torch.uint8, device=DEV)
    wp[:, :N, :K] = w.view(torch.uint8)
    xsp = torch.full((M, xs.shape[1] + 5), float("nan"), device=DEV)
    xsp[:, :xs.shape[1]] = xs
    wsp = torch.full((E, ws.shape[1] + 1, ws.shape[2] + 2), float("nan"), device=DEV)
    wsp[:, :ws.shape[1], :ws.shape[2]] = ws
    c = torch.zeros(M, ldc, dtype=torch.bfloat16, device=DEV)
    lib = _lib.load()
    size = lib.fg_grouped_block_fp8_gemm_workspace_bytes(M, N, K)
    work = torch.zeros(size, dtype=torch.uint8, device=DEV)
    st = lib.fg_grouped_block_fp8_gemm(
        xp.data_ptr(), lda, wp.data_ptr(), ldb, rows * ldb, xsp.data_ptr(), xsp.stride(0), 1, wsp.data_ptr(), wsp.stride(1), 1, wsp.stride(0),
        ends.data_ptr(), E, None, 1, M, 0, None, c.data_ptr(), ldc, _lib.DTYPE_CODE[torch.bfloat16], M, N, K, 128, 128,
        work.data_ptr(), size, _lib.current_stream_ptr(torch.device(DEV)))
    _lib.check(st, "fg_grouped_block_fp8_gemm")
    assert torch.equal(c[:, :N], base) and not c[:, N:].any()
