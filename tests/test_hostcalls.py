"""The native host side of the block GEMM and the group quantizer (csrc/hostcalls.cpp): what it takes gives the bits of the
general Python path, and whatever is not the plain case is left to that path."""
import pytest
import torch

import flag_gems
from flaggems_amd import _lib

DEV = "cuda:0"


def _pure_python(call):
    """The same call with the native functions taking nothing."""
    class Nothing:
        block_matmul = group_quant = staticmethod(lambda *a: None)

    native, _lib._host = _lib.host(), Nothing
    try:
        return call()
    finally:
        _lib._host = native


def _bits(t):
    return t.contiguous().view(torch.uint8)


def test_host_tensors_are_left_to_the_general_path():
    h, a = _lib.host(), torch.zeros(2, 128)
    assert h.block_matmul(a, a, a, a, 128, 128, torch.bfloat16, False) is None
    assert h.group_quant(a, 128, False, 1e-10, 0, 1, 0) is None
    assert h.block_matmul(None, 1, "x", a, 128, 128, torch.bfloat16, False) is None
    for beyond in (2 ** 70, -(2 ** 70)):  # fits no long: no error left behind
        assert h.block_matmul(a, a, a, a, beyond, 128, torch.bfloat16, False) is None
        assert h.block_matmul(a, a, a, a, 128, beyond, torch.bfloat16, False) is None
        assert h.group_quant(a, beyond, False, 1e-10, 0, 1, 0) is None
    with pytest.raises(TypeError):
        h.connect(1, 2)


def test_the_modules_bring_no_thread_local_storage():
    """A module with a thread-local segment that nothing touches makes every access to the thread-local storage of the libraries
    loaded before it slow (glibc before 2.39): all other host work of the process, by a sixth."""
    import struct

    from flaggems_amd.build import fastcall_path, hostcalls_path

    for path in (fastcall_path(), hostcalls_path()):
        with open(path, "rb") as f:
            data = f.read()
        assert data[:6] == b"\x7fELF\x02\x01"
        offset, = struct.unpack_from("<Q", data, 32)
        size, count = struct.unpack_from("<HH", data, 54)
        kinds = [struct.unpack_from("<I", data, offset + i * size)[0] for i in range(count)]
        assert 1 in kinds and 7 not in kinds, path  # PT_LOAD, PT_TLS


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,cols,pad", [(1, 128, 0), (5, 384, 0), (7, 1024, 64), (1, 256, 32), (300, 7168, 0)])
@pytest.mark.parametrize("columns,ue8m0", [(False, False), (True, False), (False, True)])
def test_group_quant(rows, cols, pad, dtype, columns, ue8m0):
    x = torch.randn(rows, cols + pad, device=DEV, dtype=dtype)[:, :cols]
    call = lambda: flag_gems.per_token_group_quant_fp8(x, 128, column_major_scales=columns, scale_ue8m0=ue8m0)  # noqa: E731
    rule = _lib.FG_POW2_LOG2 if ue8m0 else _lib.FG_POW2_NONE
    assert _lib.host().group_quant(x, 128, columns, 1e-10, 0, 1, rule) is not None
    (q, s), (q2, s2) = call(), _pure_python(call)
    assert q.shape == q2.shape and q.dtype == q2.dtype and q.stride() == q2.stride()
    assert s.shape == s2.shape and s.dtype == s2.dtype and s.stride() == s2.stride()
    assert torch.equal(_bits(q), _bits(q2)) and torch.equal(s, s2)


@pytest.mark.gpu
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (3, 130, 256), (17, 576, 384), (64, 4096, 1024), (300, 640, 7168)])
def test_block_matmul(M, N, K, out):
    xq, xs = flag_gems.per_token_group_quant_fp8(torch.randn(M, K, device=DEV), 128)
    w, ws = flag_gems.per_block_cast_to_fp8(torch.randn(N, K + 16, device=DEV)[:, :K], False, 128)
    forms = {"plain": (xq, w, xs, ws), "columns of scales": (xq, w, xs.t().contiguous().t(), ws), "transposed scales": (xq, w, xs, ws.t().contiguous().t()),
             "rows apart": (xq, torch.cat([w.view(torch.uint8)] * 2, 1)[:, :K].view(w.dtype), xs, ws), "parameter": (xq, torch.nn.Parameter(w, requires_grad=False), xs, ws)}
    for name, (a, b, s, t) in forms.items():
        call = lambda: flag_gems.w8a8_block_fp8_matmul(a, b, s, t, [128, 128], out)  # noqa: E731
        assert _lib.host().block_matmul(a, b, s, t, 128, 128, out, False) is not None, name
        c, c2 = call(), _pure_python(call)
        assert c.shape == c2.shape and c.dtype == c2.dtype == out and not c.requires_grad, name
        assert torch.equal(_bits(c), _bits(c2)), name
    with torch.inference_mode():
        assert torch.equal(_bits(flag_gems.w8a8_block_fp8_matmul(xq, w, xs, ws, [128, 128], out)), _bits(c))


@pytest.mark.gpu
def test_what_is_not_plain_is_left_to_the_general_path():
    h = _lib.host()
    xq, xs = flag_gems.per_token_group_quant_fp8(torch.randn(4, 256, device=DEV), 128)
    w, ws = flag_gems.per_block_cast_to_fp8(torch.randn(256, 256, device=DEV), False, 128)

    class Sub(torch.Tensor):
        pass

    for a, b, s, t, bn in ((xq[None], w, xs[None], ws, 128), (xq.as_subclass(Sub), w, xs, ws, 128), (xq[:, :128], w, xs, ws, 128), (xq, w[:, :128], xs, ws, 128),
                           (xq, w, xs[:3], ws, 128), (xq, w, xs.double(), ws, 128), (xq, w, xs, ws, 64), (xq[:0], w, xs[:0], ws, 128), (xq.cpu(), w, xs, ws, 128),
                           (xq.view(torch.int8), w, xs, ws, 128), (xq, w.t(), xs, ws, 128), (xq, w, xs, ws[:1], 128)):
        assert h.block_matmul(a, b, s, t, bn, 128, torch.bfloat16, False) is None
    assert h.block_matmul(xq, w, xs, ws, 128, 128, torch.float64, False) is None
    x = torch.randn(4, 256, device=DEV)
    for y, g in ((x[None], 128), (x.t(), 4), (x, 100), (x, 0), (x.double(), 128), (x[:0], 128), (x.as_subclass(Sub), 128), (x.int(), 128)):
        assert h.group_quant(y, g, False, 1e-10, 0, 1, 0) is None
    # and the general path's own answers
    assert flag_gems.w8a8_block_fp8_matmul(xq[None], w, xs[None], ws, [128, 128]).shape == (1, 4, 256)
    with pytest.raises(AssertionError):
        flag_gems.w8a8_block_fp8_matmul(xq, w, xs[:3], ws, [128, 128])
    with pytest.raises(AssertionError):
        flag_gems.per_token_group_quant_fp8(x, 100)
    # a group size that the kernel refuses is refused with its message, through the same exception
    for call in (lambda: flag_gems.per_token_group_quant_fp8(x, 256 + 0), lambda: flag_gems.per_token_group_quant_fp8(x, 1)):
        try:
            want = _pure_python(call)
        except Exception as e:
            with pytest.raises(type(e)):
                call()
        else:
            assert torch.equal(_bits(call()[0]), _bits(want[0]))


@pytest.mark.gpu
def test_in_a_graph_on_a_stream_of_its_own():
    M, N, K = 33, 4608, 7168  # K split: the call asks for a workspace
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w, ws = flag_gems.per_block_cast_to_fp8(torch.randn(N, K, device=DEV), False, 128)

    def step():
        xq, xs = flag_gems.per_token_group_quant_fp8(x, 128)
        return flag_gems.w8a8_block_fp8_matmul(xq, w, xs, ws, [128, 128])

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        c = step()
    for seed in range(3):
        x.copy_(torch.randn(M, K, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, step())
