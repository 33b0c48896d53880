"""The persistent grouped kernel on tiles of 64 and 128 rows, which serve few rows per group where the streaming kernel does not: more
than 64 groups of 25 - 32 rows, more than 1024 groups, 49 - 96 rows a group, and few groups with one or two K-blocks.  Tiles cut
along K, the table of tile rows, rows read through an index, scattered and weighted results, both 16-bit types."""
import pytest
import torch

import flag_gems

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
_STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}

# groups, rows a group on average, N, K
CASES = [
    (72, 28, 512, 2048),   # 64-row tiles, two cuts
    (72, 28, 520, 4096),   # four cuts; N ends inside a tile
    (66, 32, 1032, 1152),  # K-blocks that cannot be halved
    (1100, 12, 128, 2048),
    (40, 60, 384, 2048),   # 128-row tiles
    (24, 96, 264, 4096),
    (4, 10, 512, 256),     # few groups, one or two K-blocks: 64-row tiles, the groups scanned
    (3, 30, 2056, 128),    # 128-row tiles
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["sorted", "gathered", "scattered"])
@pytest.mark.parametrize("E,per,N,K", CASES)
def test_short_tiles(E, per, N, K, form, dtype):
    g = torch.Generator().manual_seed(E + N + K)
    M, top_k = E * per, 3
    weights = torch.rand(E, generator=g) + 0.4
    weights[1] = 0.0  # an empty group
    counts = torch.bincount(torch.multinomial(weights, M, True, generator=g), minlength=E)
    ends = counts.cumsum(0).int().to(DEV)
    T = M if form == "sorted" else -(-M // top_k)
    x = torch.randn(T, K, generator=g).to(torch.float8_e4m3fn).to(DEV)
    w = (0.5 * torch.randn(E, N, K, device=DEV)).to(torch.float8_e4m3fn)
    xs = (torch.rand(T, K // 128, generator=g) * 0.02 + 0.005).to(DEV)
    ws = torch.rand(E, -(-N // 128), K // 128, device=DEV) * 0.02 + 0.005
    slot = torch.randperm(M, generator=g).int()
    src = torch.arange(M, device=DEV) if form == "sorted" else (slot // top_k).long().to(DEV)
    factor = torch.ones(M, device=DEV)
    kwargs = {}
    if form != "sorted":
        kwargs = dict(row_index=slot.to(DEV), index_divisor=top_k)
    if form == "scattered":
        row_weights = (torch.rand(M, generator=g) + 0.25).to(DEV)
        kwargs.update(scatter_rows=M, row_weights=row_weights)
        factor = row_weights[slot.long().to(DEV)]
    got = flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], dtype, **kwargs)
    assert torch.equal(got, flag_gems.grouped_w8a8_block_fp8_matmul(x, w, xs, ws, ends, [128, 128], dtype, **kwargs))
    if form == "gathered":  # the same rows handed over in sorted order: the same products in the same order
        assert torch.equal(got, flag_gems.grouped_w8a8_block_fp8_matmul(x[src].contiguous(), w, xs[src].contiguous(), ws, ends, [128, 128], dtype))
    rows = got[slot.long().to(DEV)] if form == "scattered" else got
    begin = 0
    for e, end in enumerate(ends.tolist()):
        if end > begin and (E < 200 or e % 50 == 0):
            a = x[src[begin:end]].float() * xs[src[begin:end]].repeat_interleave(128, 1) * factor[begin:end, None]
            b = w[e].float() * ws[e].repeat_interleave(128, 1).repeat_interleave(128, 0)[:N]
            # half a step of the 16-bit type, twice that, plus the matrix instruction's alignment of 128 products to the largest one
            assert ((rows[begin:end].float() - a @ b.t()).abs() <= (a @ b.t()).abs() * _STEP[dtype] + 4e-4 * (a.abs() @ b.abs().t())).all()
        begin = end
