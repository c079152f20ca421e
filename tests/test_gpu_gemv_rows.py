"""One activation row against GGUF weights of any length: the GEMV that walks a row's chunks.

The kernel's operand is fp16: an fp16 row as it is, a bf16 row normalized (exactly), an fp32 row rounded once, as the
tests round it.  The codes are exact integers, so an fp32 output differs from the float64 product with that operand
by fp32 summation alone: 1e-6 of the product's own bound ||x|| ||w_n||, about ten times the 1e-7 that K = 5120
measures.  A lost or misplaced unit of 8 values moves it by sqrt(8) / K of the bound, 1.7e-4 at the longest row.
"""
import numpy as np
import pytest
import torch

import oracle as O
from gguf_blocks import random_gguf_blocks

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TYPES = ["Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K", "IQ4_NL", "IQ4_XS"]
# k, n: one chunk and one row; odd chunk counts (a ragged last step); a row past one wave's lanes;
# several row groups per wave with a ragged last group; the longest row; one chunk past it; the lengths whose fp16 rows
# another kernel keeps in registers
SIZES = [(256, 1), (768, 33), (2560, 300), (5120, 13825), (13824, 77), (16384, 130), (16640, 40), (768, 4100), (1024, 50),
         (2048, 100), (4096, 70), (8192, 36)]


def _operand(x):
    """The row that the kernel multiplies, in float64: fp32 values as fp16(x 2^-E) 2^E, 2^E above the row's maximum."""
    if x.dtype != torch.float32:
        return x.double().numpy()
    e = int(np.frexp(x.abs().max().item())[1])
    return np.ldexp(torch.ldexp(x, torch.tensor(-e)).half().double().numpy(), e)


def _limit(name, k, dtype):
    """The error a row may show, of ||x|| ||w_n||."""
    if k > 16384:  # the 16-row or the tiled kernel, whose operand may be the weight rounded to fp16
        return 5e-4
    if dtype == torch.float16 and k in ((1024, 2048, 4096) if name == "Q8_0" else (2048, 4096, 8192)):
        # codes as fp16 1024 + q, the 1024 taken off the sums: terms of 1024 |x| / |d q| times the result's, summed in
        # fp32 (about 100 for 4-bit codes near 8: 100 x 1e-7, and a margin of ten)
        return 1e-4
    return 1e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,n", SIZES)
@pytest.mark.parametrize("name", TYPES)
def test_gemv_rows(name, k, n, dtype):
    import qlin
    raw = random_gguf_blocks(name, n, k, seed=n + k)
    w = O.gguf_dequantize(raw, name, (n, k)).astype(np.float64)
    g = torch.Generator().manual_seed(k)
    x = (torch.randn(1, k, generator=g) * torch.exp(torch.randn(1, k, generator=g))).to(dtype)
    bias = torch.randn(n, generator=g)
    y = qlin.gguf_linear(x.to(DEV), torch.from_numpy(raw).to(DEV), name, (n, k), bias.to(DEV), out_dtype=torch.float32)
    xd = _operand(x)
    want = (xd @ w.T).reshape(-1) + bias.double().numpy()
    bound = np.linalg.norm(xd) * np.linalg.norm(w, axis=1) + np.abs(bias.double().numpy())
    err = np.abs(y.double().cpu().numpy().reshape(-1) - want) / bound
    assert err.max() < _limit(name, k, dtype), f"{name} k={k} n={n}: {err.max():.2e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,n", [(768, 4100), (2560, 300), (5120, 100), (13824, 77), (16384, 130)])
@pytest.mark.parametrize("name", TYPES)
def test_gemv_rows_last_values(name, k, n, dtype):
    """Only the row's last 8 values are not zero: the bound is theirs, so nothing hides a misplaced unit."""
    import qlin
    raw = random_gguf_blocks(name, n, k, seed=n + k)
    w = O.gguf_dequantize(raw, name, (n, k)).astype(np.float64)[:, -8:]
    x = torch.zeros(1, k)
    x[0, -8:] = torch.tensor([1.0, -2.0, 3.0, -5.0, 7.0, -11.0, 13.0, -17.0])  # exact in every type
    y = qlin.gguf_linear(x.to(dtype).to(DEV), torch.from_numpy(raw).to(DEV), name, (n, k), out_dtype=torch.float32)
    xd = x[0, -8:].double().numpy()
    # the K-quants' minima cancel against the codes' part: bound both by the largest weight of the row's last block
    blk = np.abs(O.gguf_dequantize(raw, name, (n, k)).astype(np.float64)[:, -256:]).max(axis=1)
    diff = np.abs(y.double().cpu().numpy().reshape(-1) - w @ xd)
    assert not diff[blk == 0].any()
    err = diff[blk > 0] / (np.linalg.norm(xd) * blk[blk > 0])
    assert err.max() < 1e-6, f"{name} k={k} n={n}: {err.max():.2e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", ["Q4_K", "Q8_0", "Q4_0"])
def test_gemv_rows_zero_and_large_rows(name, dtype):
    """A zero row gives the bias; values far above the fp16 range come back through the row exponent."""
    import qlin
    k, n = 1280, 64
    raw = random_gguf_blocks(name, n, k, seed=3)
    w = O.gguf_dequantize(raw, name, (n, k)).astype(np.float64)
    wd = torch.from_numpy(raw).to(DEV)
    bias = torch.arange(n, dtype=torch.float32)
    y = qlin.gguf_linear(torch.zeros(1, k, dtype=dtype, device=DEV), wd, name, (n, k), bias.to(DEV))
    assert torch.equal(y.cpu().float().reshape(-1), bias.to(dtype).float())
    x = (torch.randn(1, k, generator=torch.Generator().manual_seed(1)) * 1e9).to(dtype)
    y = qlin.gguf_linear(x.to(DEV), wd, name, (n, k), out_dtype=torch.float32).double().cpu().numpy()
    xd = _operand(x)
    assert np.max(np.abs(y - xd @ w.T) / (np.linalg.norm(xd) * np.linalg.norm(w, axis=1))) < 1e-6
