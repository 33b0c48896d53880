"""Results that are infinite, NaN, subnormal or next to the largest value of their type, through every kernel that stores GEMM
results.  Every row of the activations holds a single 1 and a scale of its own, so a result is one weight code times one scale and
every bit of it is determined: the product in fp32, rounded to the result's type."""
import pytest
import torch

import flag_gems

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

_SCALES = [float("inf"), float("nan"), -float("inf"), 1.0, 2.0 ** -126, 2.0 ** -133, 1.5 * 2.0 ** -130, 2.0 ** -140, 3.0 * 2.0 ** -149, 1.2e37,
           7.6e35, 3.3e38, 146.3, 2.0 ** -14, 2.0 ** -17, 1.4 * 2.0 ** -20, 3.0 * 2.0 ** -25, 0.0, -1.7]


def _problem(M, N, K, seed, integer=False):
    g = torch.Generator().manual_seed(seed)
    at = torch.randint(0, K, (M,), generator=g)
    x = torch.zeros(M, K)
    x[torch.arange(M), at] = 1.0
    scale = torch.tensor(_SCALES)[(torch.arange(M) + seed) % len(_SCALES)]
    if integer:
        w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    else:
        codes = torch.randint(0, 0x7F, (N, K), generator=g, dtype=torch.uint8) | (torch.randint(0, 2, (N, K), generator=g, dtype=torch.uint8) << 7)
        codes[codes == 0x80] = 0  # (no negative zeros: a sum with the other products' zeros is +0)
        w = codes.view(torch.float8_e4m3fn)
    return x, w, scale, at


def _same(got, want):
    got = got.cpu()
    assert got.dtype == want.dtype
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    assert torch.equal(got[ok].float(), want[ok].float())


def _products(w, at, scale):
    return w.float()[:, at].t().contiguous() * scale[:, None]


BLOCK = [(1, 2112, 512), (8, 1024, 1024), (16, 4096, 256), (24, 1024, 2048), (40, 1024, 1024), (61, 7168, 2048), (100, 4096, 1024), (300, 1024, 2048),
         (200, 16512, 1024), (300, 14400, 2176), (1000, 4608, 7168), (4100, 4104, 256)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", BLOCK)
def test_block_scales(M, N, K, dtype):
    x, w, scale, at = _problem(M, N, K, M)
    xs = torch.ones(M, K // 128)
    xs[torch.arange(M), at // 128] = scale
    got = flag_gems.w8a8_block_fp8_matmul(x.to(torch.float8_e4m3fn).to(DEV), w.to(DEV), xs.to(DEV), torch.ones(-(-N // 128), K // 128, device=DEV),
                                          [128, 128], dtype)
    _same(got, _products(w, at, scale).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,N,K", [([3, 0, 9], 512, 640), ([20, 25], 1024, 1024), ([40, 45, 40], 512, 384), ([12, 7], 512, 256),
                                        ([700, 0, 500], 1024, 512), ([30] * 70, 512, 512)])
def test_grouped(counts, N, K, dtype):
    M, E = sum(counts), len(counts)
    x, w, scale, at = _problem(M, E * N, K, M)
    xs = torch.ones(M, K // 128)
    xs[torch.arange(M), at // 128] = scale
    w = w.view(E, N, K)
    got = flag_gems.grouped_w8a8_block_fp8_matmul(x.to(torch.float8_e4m3fn).to(DEV), w.to(DEV), xs.to(DEV), torch.ones(E, -(-N // 128), K // 128, device=DEV),
                                                  torch.tensor(counts).cumsum(0).int().to(DEV), [128, 128], dtype)
    want, begin = [], 0
    for e, n in enumerate(counts):
        want.append(_products(w[e], at[begin:begin + n], scale[begin:begin + n]))
        begin += n
    _same(got, torch.cat(want).to(dtype))


@pytest.mark.parametrize("operand", [torch.float8_e4m3fn, torch.int8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 1024, 1024), (24, 2048, 1024), (33, 2048, 1024), (100, 4096, 1024), (200, 17024, 2688), (600, 4096, 4096), (2100, 4112, 512)])
def test_row_and_column_scales(M, N, K, dtype, operand):
    x, w, scale, at = _problem(M, N, K, M, integer=operand is torch.int8)
    c = torch.empty(M, N, dtype=dtype, device=DEV)
    flag_gems.cutlass_scaled_mm(c, x.to(operand).to(DEV), w.to(DEV).t(), scale[:, None].contiguous().to(DEV), torch.ones(1, N, device=DEV), None)
    _same(c, _products(w, at, scale).to(dtype))
