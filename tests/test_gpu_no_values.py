"""Linears over no values (K = 0, reachable through the C ABI alone): the output is the bias, whatever kernel a
row of that many activations takes otherwise, with a residual and without a bias too."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _view(t, rows, cols, ld):
    """A [rows, cols] descriptor of t's memory, with data also where cols is 0."""
    from qlin import _lib
    d = _lib.QlinTensor()
    d.data, d.dtype, d.ndim = t.data_ptr(), _lib._TORCH_DT[t.dtype], 2
    d.shape[0], d.shape[1], d.stride[0], d.stride[1] = rows, cols, ld, 1
    return d


def _calls(m, n, dtype, bias, residual):
    from qlin import _lib
    L = _lib.load()
    st = torch.cuda.current_stream().cuda_stream
    # the empty operands point into the middle of live allocations
    x = torch.full((m, 256), 7.0, dtype=dtype, device=DEV)[:, 128:]
    w = torch.full((n, 256), 3, dtype=torch.int8, device=DEV)[:, 128:]
    s = torch.ones(n, device=DEV)
    ws = torch.empty(1 << 26, dtype=torch.uint8, device=DEV)
    ptr = ctypes.byref
    xd, wd = _view(x, m, 0, 256), _view(w, n, 0, 256)
    sr, sc = _view(s, n, 0, 1), _view(s, n, 1, 1)
    bd = ptr(_view(bias, 1, n, n)) if bias is not None else None
    tail = (ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(st))
    for op in ("Q4_K", "Q8_0", "Q6_K", "Q2_K", "int8", "a8"):
        y = torch.full((m, n), 99.0, dtype=dtype, device=DEV)
        yd = ptr(_view(y, m, n, n))
        res = (ptr(_view(residual, m, n, n)), None) if residual is not None else ()
        if op == "int8":
            f = L.qlin_int8_linear_residual if res else L.qlin_int8_linear
            rc = f(ptr(xd), ptr(wd), ptr(sc), bd, *res, yd, 0, *tail)
        elif op == "a8":
            f = L.qlin_w4a8_linear_residual if res else L.qlin_w4a8_linear
            rc = f(ptr(xd), ptr(wd), ptr(sr), ptr(sc), None, bd, *res, yd, 4, 64, 0, *tail)
        else:
            f = L.qlin_gguf_linear_residual if res else L.qlin_gguf_linear
            t = {"Q4_K": 12, "Q8_0": 8, "Q6_K": 14, "Q2_K": 10}[op]
            rc = f(ptr(xd), ctypes.c_void_p(w.data_ptr()), t, n, 0, bd, *res, yd, *tail)
        yield op, rc, y


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 300), (3, 40), (20, 130), (100, 257), (700, 500)])
def test_no_values_give_the_bias(m, n, dtype):
    bias = torch.arange(n, device=DEV).remainder(31).to(dtype)
    res = torch.arange(m * n, device=DEV).remainder(29).reshape(m, n).to(dtype)
    for b in (bias, None):
        for r in (None, res):
            want = torch.zeros(m, n, dtype=dtype, device=DEV) + (0 if b is None else b) + (0 if r is None else r)
            for op, rc, y in _calls(m, n, dtype, b, r):
                assert rc == 0, (op, m, n)
                assert torch.equal(y, want), (op, m, n)
