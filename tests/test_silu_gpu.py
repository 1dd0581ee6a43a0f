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
    are exact): within 3 ulp of fp32 for |x| <= 80 (the library exponential
    and two roundings, of the denominator and the quotient), and within 1e-30
    of the exact value, with no NaN, beyond."""
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


def _silu_of(x32, m):
    """The fused SiLU of fp32 values x32 (1-D, on the CPU), as an [m, len] result.
    Each value goes to a W row as up to three bf16 pieces that A, all ones,
    adds up exactly; the up projection is 1."""
    pieces, rest = [], x32.clone()
    for _ in range(3):
        # Truncated, so every partial sum is a prefix of x's bits.
        p = (rest.view(torch.int32) & -65536).view(F32)
        pieces.append(p)
        rest = torch.where(torch.isfinite(x32), rest - p, torch.zeros(()))
    n = x32.numel()
    w = torch.zeros((2 * n, 64))
    w[:n, 0], w[:n, 1], w[:n, 2] = pieces
    w[n:, 3] = 1
    a = torch.zeros((m, 64))
    a[:, :4] = 1
    return G.gemm_silu_mul(a.to(BF16).to(DEV), w.to(BF16).to(DEV), F32).cpu()


# Rows on splitk_decode, on the small tiles and on the large ones.
@pytest.mark.parametrize("m", [4, 40, 300])
def test_silu_bits(m):
    """x / (1 + e^-x) bit for bit as the fp32 library exponential and an IEEE
    division give it, on fp32 values of every magnitude (2^-60 to 2^127, most
    of them where e^-x counts)."""
    gen = torch.Generator().manual_seed(m)
    x = torch.cat([torch.randn(3000, generator=gen) * s for s in (0.1, 1.0, 4.0, 30.0, 100.0)])
    x = torch.cat([x, torch.ldexp(1 + torch.rand(2000, generator=gen), torch.randint(-60, 127, (2000,), generator=gen)),
                   torch.tensor([-87.3, -87.34, -88.0, -88.7, -88.72, -88.73, -104.0, 2.0 ** 126, 3.4e38, -3.4e38])])
    x = torch.where(x.abs() < 2.0 ** -60, torch.ones(()), x).float()
    _say(f"silu bits, M={m}, {x.numel()} fp32 values")
    got = _silu_of(x, m)
    with np.errstate(over="ignore"):
        want = torch.from_numpy(x.numpy() / (np.float32(1) + torch.exp(-x.to(DEV)).cpu().numpy()))
    bad = got.view(torch.int32) != want.view(torch.int32)
    assert not bool(bad.any()), f"{int(bad.sum())} of {bad.numel()} differ, e.g. at {x[bad.any(0)][:4].tolist()}"


@pytest.mark.parametrize("m", [4, 40, 300])
def test_silu_infinities_and_nan(m):
    """-inf / inf is NaN, +inf stays, NaN stays, and neighbours are untouched."""
    inf, nan = float("inf"), float("nan")
    x = torch.tensor([1.0, inf, 2.0, -inf, 3.0, nan, -1.0] * 5)
    _say(f"silu of infinities and NaN, M={m}")
    got = _silu_of(x, m)
    want = torch.tensor([1 / (1 + np.exp(-1.0)), inf, 2 / (1 + np.exp(-2.0)), nan, 3 / (1 + np.exp(-3.0)), nan,
                         -1 / (1 + np.exp(1.0))] * 5, dtype=F32).expand(m, -1)
    assert torch.allclose(got, want, rtol=1e-6, atol=0, equal_nan=True)
