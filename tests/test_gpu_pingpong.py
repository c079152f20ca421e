"""The 256 x 256 tile GEMMs whose two wave groups take turns: contractions of one k-tile up (an odd and an
even number of them, fewer than the pipeline is deep), ragged last tiles in both directions.

fp16 operands are exact here (small integers times powers of two), so the weight-only outputs differ
from the float64 product by the fp32 sum alone: 1e-6 of it relative to |x| |w|.  The A8 output is
replayed exactly: the int8 products summed in float64, then the epilogue's fp32 steps.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _ints(shape, lo, hi, seed):
    return torch.randint(lo, hi + 1, shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def _check(y, x, w, extra=None):
    want = x.double() @ w.double().T
    bound = x.double().norm(dim=1, keepdim=True) * w.double().norm(dim=1) + 1e-30
    if extra is not None:
        want = want + extra
    assert ((y.double() - want).abs() / bound).max().item() < 1e-6


@pytest.mark.parametrize("m,n", [(2305, 2600), (600, 8200)])  # 110 and 99 tiles, last ones 1 row, 40 and 88 x 8
@pytest.mark.parametrize("k", [64, 128, 192, 320, 1088])
def test_decoded_gguf(k, m, n):
    import qlin
    x = _ints((m, k), -8, 8, k).half()
    q = _ints((n, k), -127, 127, m).to(torch.int8)
    d = torch.full((n, k // 32, 1), 2.0 ** -7, dtype=torch.float16, device=DEV)
    raw = torch.cat([d.view(torch.uint8), q.view(n, k // 32, 32).view(torch.uint8)], 2).reshape(n, -1).contiguous()
    r = _ints((m, n), -4, 4, 7).float()
    y = qlin.gguf_linear(x, raw, "Q8_0", (n, k), out_dtype=torch.float32)
    _check(y, x, q.float() / 128)
    y = qlin.gguf_linear(x, raw, "Q8_0", (n, k), out_dtype=torch.float32, residual=r)
    _check(y, x, q.float() / 128, r.double())


@pytest.mark.parametrize("m,n", [(3329, 3000), (513, 14000)])  # 168 and 165 tiles
@pytest.mark.parametrize("k", [64, 128, 256, 384, 640, 1152])  # 64: rows of half a weight half-tile
def test_int8(k, m, n):
    import qlin
    x = _ints((m, k), -8, 8, k).half()
    q = _ints((n, k), -128, 127, m).to(torch.int8)
    y = qlin.int8_linear(x, q, torch.full((n,), 0.5, device=DEV), out_dtype=torch.float32)
    _check(y, x, q.float() / 2)


@pytest.mark.parametrize("m,n", [(3585, 3500), (600, 16400)])  # 210 and 195 tiles
@pytest.mark.parametrize("bits,k", [(4, 128), (6, 256), (4, 384), (6, 640), (4, 3584), (6, 3712)])  # two groups from 3584
def test_a8(bits, k, m, n):
    import qlin
    from qlin.quantize import pack_codes
    g = torch.Generator().manual_seed(k)
    x = torch.randn(m, k, generator=g).half().to(DEV)
    codes = torch.randint(1, 1 << bits, (n, k), generator=g)
    packed = pack_codes(codes, bits).to(DEV)
    s_rel = (1 + 3 * torch.rand(n, k // 64, generator=g)).half().to(DEV)
    s_ch = (torch.rand(n, generator=g) * 1e-2).to(DEV)
    bias = torch.randn(n, generator=g).to(DEV)
    y = qlin.w4a8_int8_linear(x, packed, s_rel, s_ch, None, None, bias, 64, 128)
    q, sx = qlin.quantize_int8_rowwise(x, 128)
    acc = q.double() @ qlin.w4a8_int8_grid(packed, s_rel, None, 64).double().T
    want = ((acc.float() * sx) * s_ch + bias).half()
    assert torch.equal(y, want)


@pytest.mark.parametrize("m,k", [(1, 16), (129, 528)])  # columns and rows of a tile past the matrix
@pytest.mark.parametrize("n", [1, 63, 65, 129, 256, 300, 513, 900])  # 2 to 16 stages of 64, the last of them ragged
def test_grad_input(n, m, k):
    import qlin
    dy = _ints((m, n), -8, 8, n).half()
    q = _ints((n, k), -128, 127, m).to(torch.int8)
    dx = qlin.int8_linear_grad_input(dy, q, torch.full((n,), 0.5, device=DEV), False, 256, out_dtype=torch.float32)
    _check(dx, dy, q.float().T / 2)


# 306, 442 and 561 tiles, rows and columns of the last ones past the matrix: the kernel that two workgroups share a CU
# with up to 26, 32 and 36 stages of 64, and the one past them
@pytest.mark.parametrize("m,n", [(2200, 1), (2200, 129), (2200, 300), (2200, 1664), (2200, 1665), (3300, 2048), (3300, 2049),
                                 (4100, 2304), (4100, 2305)])
def test_grad_input_rounds(m, n):
    test_grad_input(n, m, 4112)


@pytest.mark.parametrize("qtype,k", [("Q8_0", 8224), ("Q8_0", 16384), ("Q6_K", 8448), ("Q6_K", 16640)])
def test_wide_rows_decoded(qtype, k):
    """Rows on both sides of the limits of the decode that keeps a row in registers (8192, 16384)."""
    import qlin
    n, m, ts, qk = 520, 1100, *{"Q8_0": (34, 32), "Q6_K": (210, 256)}[qtype]
    raw = _ints((n, k // qk, ts), 0, 255, k).to(torch.uint8)
    d = torch.full((n, k // qk, 1), 2.0 ** -7, dtype=torch.float16, device=DEV).view(torch.uint8)
    if qtype == "Q8_0":
        raw[:, :, :2] = d
    else:
        raw[:, :, 208:] = d
        raw[:, :, 192:208] = _ints((n, k // qk, 16), 1, 4, 5).to(torch.uint8)
    raw = raw.reshape(n, -1).contiguous()
    x = _ints((m, k), -8, 8, k).half()
    w = qlin.dequantize_gguf(raw, qtype, (n, k))  # at most 8 significant bits: exact in fp16
    _check(qlin.gguf_linear(x, raw, qtype, (n, k), out_dtype=torch.float32), x, w)


@pytest.mark.parametrize("m,n", [(1025, 16384), (1090, 16300), (2100, 8100)])  # rests of 1, 66 and 52 rows: 32- and 64-row tiles
@pytest.mark.parametrize("k", [64, 384, 512])
def test_int8_rest(k, m, n):
    """Whole rounds of 256 x 256 tiles, then the last rows through the ring kernel."""
    import qlin
    x = _ints((m, k), -8, 8, k).half()
    q = _ints((n, k), -128, 127, m).to(torch.int8)
    r = _ints((m, n), -4, 4, 7).float()
    s = torch.full((n,), 0.5, device=DEV)
    _check(qlin.int8_linear(x, q, s, out_dtype=torch.float32), x, q.float() / 2)
    _check(qlin.int8_linear(x, q, s, out_dtype=torch.float32, residual=r), x, q.float() / 2, r.double())


@pytest.mark.parametrize("m", [2049, 2148, 2305, 2500])  # rests of 1, 100, 257 and 452 rows: 64, 64, 128 and 128 columns
def test_a8_rest(m):
    test_a8(4, 256, m, 8192)
    test_a8(4, 3584, m, 8192)
