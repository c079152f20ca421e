"""One activation row against GGUF weights of any length: the GEMV that walks a row's chunks.

bf16 rows are exact in the kernel's normalized fp16 and the codes are exact integers, so an fp32
output differs from the float64 product by fp32 summation alone: 1e-6 of the product's own bound
||x|| ||w_n||, about ten times the 1e-7 that K = 5120 measures.  fp16 and fp32 rows add the rounding
of x to fp16 (2^-11 of each value, so 5e-4 of the bound).
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
# several row groups per wave with a ragged last group; the longest row; one chunk past it
SIZES = [(256, 1), (768, 33), (2560, 300), (5120, 13825), (13824, 77), (16384, 130), (16640, 40)]


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
    xd = x.double().numpy()
    want = (xd @ w.T).reshape(-1) + bias.double().numpy()
    bound = np.linalg.norm(xd) * np.linalg.norm(w, axis=1) + np.abs(bias.double().numpy())
    err = np.abs(y.double().cpu().numpy().reshape(-1) - want) / bound
    # past 16384 another kernel takes the row, whose operand may be the weight rounded to fp16
    assert err.max() < (1e-6 if dtype == torch.bfloat16 and k <= 16384 else 5e-4), f"{name} k={k} n={n}: {err.max():.2e}"


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
    xd = x.double().numpy()
    assert np.max(np.abs(y - xd @ w.T) / (np.linalg.norm(xd) * np.linalg.norm(w, axis=1))) < 5e-4
