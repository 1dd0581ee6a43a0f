"""GPU test of the SiLU of the fused gate/up epilogues on every input value."""
from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from test_gemm_gpu import DEV, NAME, _say

pytestmark = pytest.mark.gpu

G = importlib.import_module("inference_systems_amd.kernels.gemm")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "f16"])
def test_silu_every_input(dtype):
    """The fused SiLU on every finite value of the input type (W picks column
    0 as the gate and column 1, all ones, as the up projection, so the sums
    are exact): within 3 ulp of fp32 for |x| <= 80 (hardware exponential and
    reciprocal, 1 ulp each, and three roundings), and within 1e-30 of the
    exact value, with no NaN, beyond."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype)
    x = x[torch.isfinite(x.float())]
    a = torch.zeros((x.numel(), 64), dtype=dtype)
    a[:, 0], a[:, 1] = x, 1
    w = torch.zeros((64, 64), dtype=dtype)
    w[:32, 0], w[32:, 1] = 1, 1
    _say(f"silu on every finite {NAME[dtype]}")
    got = G.gemm_silu_mul(a.to(DEV), w.to(DEV), F32)[:, 7].cpu().double().numpy()
    x64 = x.double().numpy()
    with np.errstate(over="ignore"):
        ref = x64 / (1.0 + np.exp(-x64))
    err = np.abs(got - ref)
    normal = (np.abs(x64) <= 80) & (np.abs(ref) >= np.finfo(np.float32).tiny)
    ulp = err[normal] / np.spacing(np.abs(ref[normal]).astype(np.float32)).astype(np.float64)
    assert ulp.max() <= 3.0, f"{ulp.max():.2f} ulp at {x64[normal][ulp.argmax()]}"
    rest = ~normal
    assert (err[rest] <= 1e-30 + 1e-6 * np.abs(ref[rest])).all()
