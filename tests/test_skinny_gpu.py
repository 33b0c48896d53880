"""The kernel for few rows or few tiles (csrc/fp8_gemm_skinny.hip): every tile shape at the fewest and most rows it takes, weights that
end inside a tile, odd and even numbers of K-blocks (the last stage holds one), K in one range and split (all of them for block scales
and for row and column scales: tests/test_dispatch_rules.py asks the planner), both layouts of the activation scales, every result and
operand type."""
import pytest
import torch

import flag_gems

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

_STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}

# (rows, weight rows, K); tests/test_dispatch_rules.py holds every list against the planner: what each shape is here for
BLOCK_SCALES = [
    # 16 rows a tile: 32, 64 and 128 weight rows; short K, one round that fills the units
    (1, 512, 512), (16, 4097, 640), (5, 577, 896), (9, 6209, 1152), (1, 8192, 4096),
    (16, 12353, 1152), (1, 8194, 512),
    (16, 24641, 4224), (3, 28672, 4096), (1, 24659, 4096),
    # the same, K split
    (9, 833, 9344), (16, 1536, 14080), (13, 2500, 16512), (16, 4096, 14336), (13, 3585, 10368), (9, 513, 16512),
    (13, 1447, 16896), (13, 1350, 18048),
    (13, 3605, 20224), (11, 3598, 19584),
    # 32 rows a tile
    (17, 8129, 1152), (32, 7105, 768), (20, 3000, 768), (17, 1030, 14336), (22, 1028, 11392),
    (32, 12290, 1280), (17, 16523, 512), (29, 8194, 640), (19, 1359, 13056), (25, 1772, 11136),
    (31, 28609, 1152), (17, 16742, 1280), (32, 4100, 14464), (17, 4354, 10240),
    # 64 rows a tile
    (33, 7105, 1152), (64, 7105, 1152), (61, 640, 512), (33, 2701, 10496), (35, 1623, 13952),
    (33, 8234, 512), (56, 8715, 640), (64, 4097, 8064), (48, 1600, 11008), (33, 2100, 9856),
    (63, 28609, 1152), (33, 16734, 512), (64, 7168, 16384), (43, 5555, 8832),
    # 128 rows a tile
    (65, 3073, 3200), (128, 14337, 1152), (67, 8290, 512), (127, 4100, 7552), (97, 2112, 7168),
    # several rows of tiles, the last of one row, of a part and full: 64 x 32
    (1001, 128, 512), (1019, 128, 640), (321, 577, 5248), (449, 512, 8064), (1001, 128, 2688), (129, 775, 3072),
    # 64 x 64
    (4096, 129, 896), (193, 2049, 512), (130, 3073, 2560), (129, 2100, 5248), (257, 1537, 5120), (191, 1537, 12288),
    # 64 x 128
    (193, 4100, 512), (257, 6209, 7168), (321, 3073, 896), (129, 2049, 7168), (257, 2049, 8192), (130, 1828, 6272),
    # 128 x 64
    (193, 4100, 2688), (513, 3073, 2560), (1000, 577, 8192), (385, 1537, 8064), (204, 1348, 5760),
]
# (rows of the result are multiples of 16 bytes here; 16 rows a tile are not split along K)
ROW_AND_COLUMN_SCALES = [
    (1, 512, 512), (16, 4112, 640), (5, 592, 896), (9, 8192, 8192), (16, 8176, 8192),
    (16, 12368, 1152), (1, 8208, 512),
    (16, 24656, 1152), (3, 28672, 4096), (1, 24672, 4096),
    (17, 8144, 1152), (32, 7120, 768), (20, 3008, 768), (17, 1040, 14336), (22, 1040, 11392),
    (32, 12304, 1280), (17, 16528, 512), (29, 8208, 640), (19, 1360, 13056), (25, 1776, 11136),
    (31, 28624, 1152), (17, 16752, 1280), (32, 4112, 14464), (17, 4368, 10240),
    (33, 7120, 1152), (64, 7120, 1152), (61, 640, 512), (33, 2704, 10496), (35, 1632, 13952),
    (33, 8240, 512), (56, 8720, 640), (64, 4112, 8064), (48, 1600, 11008), (33, 2112, 9856),
    (63, 28624, 1152), (33, 16736, 512), (64, 7168, 16384), (33, 5664, 11392),
    (65, 3088, 3200), (128, 14352, 1152), (67, 8304, 512), (127, 4112, 7552), (97, 2112, 7168), (100, 5008, 16384),
    (1001, 128, 512), (1019, 128, 640), (321, 592, 5248), (449, 512, 8064), (1001, 128, 2688), (129, 784, 3072),
    (4096, 144, 896), (193, 2064, 512), (130, 3088, 2560), (129, 1056, 4736), (135, 976, 5120), (191, 1552, 12288),
    (193, 4112, 512), (257, 6224, 8192), (321, 3088, 896), (130, 1936, 10240), (130, 2752, 5248), (257, 2064, 8192),
    (193, 4112, 2688), (513, 3088, 2560), (1000, 592, 8192), (200, 1072, 8576), (385, 1552, 8064),
]


@pytest.mark.parametrize("columns_of_scales", [False, True])
@pytest.mark.parametrize("M,N,K", BLOCK_SCALES)
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


@pytest.mark.parametrize("result", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", ROW_AND_COLUMN_SCALES)
def test_row_and_column_scales(M, N, K, result):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g, device=DEV) * 20).to(torch.float8_e4m3fn)
    w = (torch.randn(N, K, generator=g, device=DEV) * 20).to(torch.float8_e4m3fn)
    sa, sb = torch.rand(M, 1, generator=g, device=DEV) * 0.01, torch.rand(1, N, generator=g, device=DEV) * 0.01
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    c = torch.empty(M, N, device=DEV, dtype=result)
    flag_gems.cutlass_scaled_mm(c, x, w.t(), sa, sb, bias)
    a, b = x.float(), w.float()
    want, mag = (a @ b.t()) * sa * sb + bias.float(), (a.abs() @ b.abs().t()) * sa * sb + bias.float().abs()
    # (the bias is added to the rounded product: one more rounding, of a value no larger than mag's terms)
    assert ((c.float() - want).abs() <= (want.abs() + (want - bias.float()).abs()) * _STEP[result] + 4e-4 * mag).all()


@pytest.mark.parametrize("result", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", ROW_AND_COLUMN_SCALES)
def test_int8_products_are_exact(M, N, K, result):
    """The sums are whole numbers below 2^31, whatever the order of the groups and splits; then one rounding to float, the two
    scales, one rounding to the result's type, and the bias with another."""
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g, device=DEV) * 60).clamp(-127, 127).to(torch.int8)
    w = (torch.randn(N, K, generator=g, device=DEV) * 60).clamp(-127, 127).to(torch.int8)
    sa, sb = torch.rand(M, 1, generator=g, device=DEV) * 0.01, torch.rand(1, N, generator=g, device=DEV) * 0.01
    sums = (x.double() @ w.double().t()).float()  # exact in double
    for bias in (None, torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)):
        c = torch.empty(M, N, device=DEV, dtype=result)
        flag_gems.cutlass_scaled_mm(c, x, w.t(), sa, sb, bias)
        want = ((sums * sa) * sb).to(result)
        if bias is not None:
            want = (want.float() + bias.float()).to(result)
        assert torch.equal(c, want)


# a shape of every tile, K in one range and split
_EVERY_TILE = [(16, 4097, 640), (16, 1536, 14080), (16, 12353, 1152), (13, 1447, 16896), (16, 24641, 4224), (13, 3605, 20224),
               (17, 8129, 1152), (17, 1030, 14336), (32, 12290, 1280), (19, 1359, 13056), (31, 28609, 1152), (32, 4100, 14464),
               (33, 7105, 1152), (33, 2701, 10496), (33, 8234, 512), (64, 4097, 8064), (63, 28609, 1152), (64, 7168, 16384),
               (128, 14337, 1152), (127, 4100, 7552), (321, 577, 5248), (130, 3073, 2560), (129, 2049, 7168), (193, 4100, 2688)]


@pytest.mark.parametrize("M,N,K", _EVERY_TILE)
def test_rows_further_apart_than_they_are_long(M, N, K):
    """Activations, weights, scales and results in the middle of wider matrices: the bits of the call on matrices of their own, and
    nothing beside the result is written."""
    from flaggems_amd import _lib
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.float8_e4m3fn)
    xs = torch.rand(M, K // 128, generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(-(-N // 128), K // 128, generator=g, device=DEV) * 0.02 + 0.005
    want = flag_gems.w8a8_block_fp8_matmul(x, w, xs, ws, [128, 128])

    def apart(t, pad):  # rows with `pad` values on either side
        wide = torch.zeros(t.shape[0], t.shape[1] + 2 * pad, dtype=t.dtype, device=DEV)
        part = wide[:, pad:pad + t.shape[1]]
        part.copy_(t)
        return part

    x, w, xs, ws = apart(x, 48), apart(w, 16), apart(xs, 3), apart(ws, 5)
    wide = torch.full((M, N + 32), 7.0, dtype=torch.bfloat16, device=DEV)
    c = wide[:, 16:16 + N]
    lib, dev = _lib.load(), torch.device(DEV)
    wsp = _lib.workspace(dev, lib.fg_block_fp8_gemm_workspace_bytes(M, N, K))
    rc = lib.fg_block_fp8_gemm(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), xs.data_ptr(), xs.stride(0), 1, ws.data_ptr(), ws.stride(0), 1,
                               c.data_ptr(), c.stride(0), _lib.FG_BF16, M, N, K, 128, 128, wsp.data_ptr(), wsp.numel(), _lib.current_stream_ptr(dev))
    _lib.check(rc, "fg_block_fp8_gemm")
    assert torch.equal(c, want)
    assert (wide[:, :16] == 7.0).all() and (wide[:, 16 + N:] == 7.0).all()


# what other kernels serve: calls without the workspace that a split K needs (up to 16 rows, and 33 to 64 against weights that those
# kernels split too, such a call is refused), activation scales whose rows lie too far apart for
# 32-bit offsets, and K below 512 against wide weights
WITHOUT_WORKSPACE = [(17, 2304, 16384), (32, 3590, 18944), (24, 4096, 14336), (40, 19178, 8192), (65, 2112, 7168), (128, 4096, 4096), (128, 2048, 16384), (200, 1030, 4096), (190, 1280, 8192), (257, 1537, 5120)]
SCALES_FAR_APART = [(9, 3590, 18944), (16, 28672, 4096), (16, 8192, 8192), (17, 24576, 1536), (32, 28672, 4096), (24, 16384, 1024), (20, 4608, 7168),
                    (40, 24584, 1536), (33, 49152, 2048), (37, 16384, 1024), (48, 8330, 6144), (64, 6650, 8192), (50, 7168, 16384), (61, 4608, 7168)]
SHORT_K = [(40, 16384, 384), (64, 20000, 256), (24, 24576, 384), (50, 10000, 128), (60, 12345, 384), (17, 30000, 256)]


@pytest.mark.parametrize("M,N,K,how", [s + ("no workspace",) for s in WITHOUT_WORKSPACE] + [s + ("scales far apart",) for s in SCALES_FAR_APART] +
                         [s + ("",) for s in SHORT_K])
def test_calls_that_the_deep_stage_kernel_cannot_take(M, N, K, how):
    from flaggems_amd import _lib
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.float8_e4m3fn)
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.float8_e4m3fn)
    xs = torch.rand(M, K // 128, generator=g, device=DEV) * 0.02 + 0.005
    ws = torch.rand(-(-N // 128), K // 128, generator=g, device=DEV) * 0.02 + 0.005
    a = x.float() * xs.repeat_interleave(128, 1)
    b = w.float() * ws.repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]
    want, mag = a @ b.t(), a.abs() @ b.abs().t()
    lib, dev = _lib.load(), torch.device(DEV)
    if how == "scales far apart":
        far = torch.zeros(M, 1 << 21, device=DEV)
        far[:, :K // 128] = xs
        xs = far[:, :K // 128]
    for dtype in _STEP:
        wsp = None if how == "no workspace" else _lib.workspace(dev, lib.fg_block_fp8_gemm_workspace_bytes(M, N, K))
        got = []
        for _ in range(2):
            c = torch.full((M, N), 7.0, device=DEV, dtype=dtype)
            rc = lib.fg_block_fp8_gemm(x.data_ptr(), K, w.data_ptr(), K, xs.data_ptr(), xs.stride(0), 1, ws.data_ptr(), ws.stride(0), 1, c.data_ptr(), N,
                                       _lib.DTYPE_CODE[dtype], M, N, K, 128, 128, None if wsp is None else wsp.data_ptr(), 0 if wsp is None else wsp.numel(),
                                       _lib.current_stream_ptr(dev))
            _lib.check(rc, "fg_block_fp8_gemm")
            got.append(c)
        assert ((got[0].float() - want).abs() <= want.abs() * _STEP[dtype] + 4e-4 * mag).all()
        assert torch.equal(*got)


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
