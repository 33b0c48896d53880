"""The 256 x 128 tiles of the deep-pipelined tile kernel (csrc/fp8_gemm.hip): problems with more 128-row tiles than compute
units but no more 256-row ones.  Edges: the fewest rows and columns that take it, a row past a tile, ragged N, the shortest and
the longest K of the rule, every result type and operand type."""
import pytest
import torch

import flag_gems

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


_STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _close(got, want, mag):
    # half a step of the result's type (2^-9 of the value for bf16), twice that, plus the matrix instruction's alignment of 128
    # products to the largest one: below 2e-4 of the sum of |a||b|
    assert ((got.float() - want).abs() <= want.abs() * _STEP[got.dtype] + 4e-4 * mag).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(129, 16513, 1024), (256, 16600, 1152), (257, 11016, 1152), (511, 8320, 1024), (1000, 4608, 2304), (300, 16384, 8192), (129, 16513, 896)])
def test_block_scales(M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.float8_e4m3fn)
    xs = torch.rand(M, K // 128, generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(-(-N // 128), K // 128, generator=g, device=DEV) * 0.02 + 0.005
    got = flag_gems.w8a8_block_fp8_matmul(x, w, xs, ws, [128, 128], dtype)
    a = x.float() * xs.repeat_interleave(128, 1)
    b = w.float() * ws.repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]
    assert got.dtype == dtype
    _close(got, a @ b.t(), a.abs() @ b.abs().t())


@pytest.mark.parametrize("operand", [torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("M,N,K", [(129, 16640, 1024), (500, 10240, 1280), (257, 11024, 1152),
                                   # the first three go to 128-row tiles, as row and column scales with short K are faster there; these do not
                                   (129, 19072, 2176), (256, 16512, 2688), (511, 9600, 3200), (129, 20480, 4224)])
def test_row_and_column_scales(M, N, K, operand):
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
