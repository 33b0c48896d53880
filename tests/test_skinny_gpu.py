"""The kernel for few rows or few tiles (csrc/fp8_gemm_skinny.hip): every tile shape at the fewest and most rows it takes, weights that
end inside a tile, odd and even numbers of K-blocks (the last stage holds one), K in one range and split, both layouts of the
activation scales, every result and operand type."""
import pytest
import torch

import flag_gems

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

_STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}

_SHAPES = [
    # 16 rows a tile: 32, 64 and 128 weight rows; short K, one round that fills the units
    (1, 512, 512), (16, 4097, 640), (5, 577, 896), (9, 6209, 1152), (16, 12353, 1152), (16, 24641, 1152), (3, 28672, 4096), (1, 8192, 4096),
    # K split
    (9, 833, 9344), (16, 1536, 14080), (13, 2500, 16512), (16, 4096, 14336), (13, 3585, 10368), (9, 513, 16512),
    # 32 rows a tile
    (17, 8129, 1152), (32, 12290, 1280), (31, 28609, 1152), (17, 1030, 14336), (32, 4100, 14464), (20, 3000, 768),
    # 64 rows a tile
    (33, 7105, 1152), (64, 4097, 8064), (63, 28609, 1152), (64, 7168, 16384), (33, 2100, 9856), (48, 1600, 11008), (61, 640, 512),
    # 128 rows a tile
    (65, 3073, 1152), (128, 14337, 1152), (127, 4100, 7552), (97, 2112, 7168),
    # several rows of tiles, the last of one row, of a part and full: 64 x 32
    (1001, 128, 512), (4096, 129, 896), (321, 577, 5248), (449, 512, 8064), (1001, 128, 2688),
    # 64 x 64
    (193, 2049, 512), (130, 3073, 2560), (129, 2100, 5248), (257, 1537, 5120), (191, 1537, 12288),
    # 64 x 128
    (193, 4100, 512), (257, 6209, 7168), (321, 3073, 896), (129, 2049, 7168), (257, 2049, 8192),
    # 128 x 64
    (193, 4100, 2688), (513, 3073, 2560), (1000, 577, 8192), (385, 1537, 8064),
]


@pytest.mark.parametrize("columns_of_scales", [False, True])
@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_block_scales(M, N, K, columns_of_scales):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.float8_e4m3fn)
    xs = torch.rand(M, K // 128, generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(-(-N // 128), K // 128, generator=g, device=DEV) * 0.02 + 0.005
    a = x.float() * xs.repeat_interleave(128, 1)
    b = w.float() * ws.repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]
    want, mag = a @ b.t(), a.abs() @ b.abs().t()
    if columns_of_scales:
        xs = xs.t().contiguous().t()
    for dtype in _STEP:
        got = flag_gems.w8a8_block_fp8_matmul(x, w, xs, ws, [128, 128], dtype)
        # a step of the result's type, and the matrix instruction's alignment of 128 products to the largest one: below 2e-4 of
        # the sum of |a||b|, twice that
        assert got.dtype == dtype and ((got.float() - want).abs() <= want.abs() * _STEP[dtype] + 4e-4 * mag).all()
        # whichever block comes last adds the parts of K in their order
        assert torch.equal(got, flag_gems.w8a8_block_fp8_matmul(x, w, xs, ws, [128, 128], dtype))


@pytest.mark.parametrize("operand", [torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("M,N,K", _SHAPES + [(100, 5000, 16384)])
def test_row_and_column_scales(M, N, K, operand):
    N = -(-N // 16) * 16  # (rows of the result must be multiples of 16 bytes here)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g, device=DEV) * 20).clamp(-127, 127).to(operand)
    w = (torch.randn(N, K, generator=g, device=DEV) * 20).clamp(-127, 127).to(operand)
    sa, sb = torch.rand(M, 1, generator=g, device=DEV) * 0.01, torch.rand(1, N, generator=g, device=DEV) * 0.01
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    c = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    flag_gems.cutlass_scaled_mm(c, x, w.t(), sa, sb, bias)
    a, b = x.float(), w.float()
    want, mag = (a @ b.t()) * sa * sb + bias.float(), (a.abs() @ b.abs().t()) * sa * sb + bias.float().abs()
    # (the bias is added to the rounded product: one more rounding, of a value no larger than mag's terms)
    assert ((c.float() - want).abs() <= (want.abs() + (want - bias.float()).abs()) * 2.0 ** -8 + 4e-4 * mag).all()


def test_rows_past_the_last_do_not_reach_the_result():
    # one row of a 16- and of a 64-row tile whose other rows are whatever the kernel before left in LDS: NaN codes
    N, K = 8192, 4096
    w = torch.randn(N, K, device=DEV).to(torch.float8_e4m3fn)
    ws = torch.ones(N // 128, K // 128, device=DEV)
    nan = torch.full((256, K), float("nan"), device=DEV).to(torch.float8_e4m3fn)
    for rows in (1, 17, 33, 65, 193):
        x = torch.randn(rows, K, device=DEV).to(torch.float8_e4m3fn)
        flag_gems.w8a8_block_fp8_matmul(nan, w, torch.ones(256, K // 128, device=DEV), ws, [128, 128])
        got = flag_gems.w8a8_block_fp8_matmul(x, w, torch.ones(rows, K // 128, device=DEV), ws, [128, 128])
        assert not got.isnan().any()
