"""GPU tests of mfma_staged's 128-row tiles for about one round on the CUs
(csrc/gemm_mid.hip): grids that take them at the edges of tiles, K-tiles and the
C tile's store, against the same rows computed 100 at a time (smaller tiles, which
sum K in the same order, so every bit is equal) and against the oracle."""
from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, NAME, _check_silu_mul, _check_tolerance, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
K = importlib.import_module("inference_systems_amd.kernels.prologue")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _inputs(m, rows, k, dtype):
    gen = torch.Generator().manual_seed(m + rows + k)
    return torch.randn((m, k), generator=gen).to(dtype), (torch.randn((rows, k), generator=gen) * 0.1).to(dtype)


# 128 x 256 tiles: 133 to 252 of them, and more than 512 (two rounds and a part);
# 128 x 128: 144 and 210.  N = 4333 / 2001 store element by element at the end of
# rows (and, with 2-byte outputs, everywhere); K = 256 / 264 / 328 / 384 / 456 is
# 4-8 K-tiles with tails of 0, 8, 8, 0 and 8.
@pytest.mark.parametrize("m,n,k,din,dout", [
    (1000, 4333, 264, BF16, BF16), (1000, 4333, 328, F16, F32), (1801, 4096, 256, BF16, BF16),
    (2300, 3333, 384, BF16, F32), (3000, 6144, 456, BF16, BF16), (2200, 1001, 264, BF16, F32),
    (1100, 2001, 328, F16, F16), (1792, 1920, 456, BF16, BF16)], ids=lambda v: NAME.get(v, v))
def test_mid_tiles(m, n, k, din, dout):
    a, w = _inputs(m, n, k, din)
    ad, wd = a.to(DEV), w.to(DEV)
    _say(f"mid M={m} N={n} K={k} {NAME[din]}->{NAME[dout]}")
    out = G.gemm_with_kernel(ad, wd, L.KERNEL_MFMA_STAGED, dout)
    assert L.last_kernel() == f"mfma_mid 128x{128 if n in (1001, 2001, 1920) else 256}"
    for r0 in (0, 100, m - 200, m - 100):
        part = G.gemm_with_kernel(ad[r0:r0 + 100], wd, L.KERNEL_MFMA_STAGED, dout)
        torch.cuda.synchronize()
        assert torch.equal(out[r0:r0 + 100], part), f"rows {r0}: {int((out[r0:r0 + 100] != part).sum())} outputs differ"
    rows = np.array([0, 63, 64, 127, 128, m - 1])
    _check_tolerance(out.cpu(), a, w, L.B_NK, dout, rows=rows)


@pytest.mark.parametrize("norm", [False, True], ids=["plain", "add-norm"])
@pytest.mark.parametrize("dout", [BF16, F32], ids=["bf16", "f32"])
def test_mid_tiles_silu(norm, dout):
    """Gate/up pairs and the row scale of the norm: 12 x 18 tiles, ragged in
    both directions."""
    m, n, k = 1500, 2203, 264
    a, w = _inputs(m, 2 * n, k, BF16)
    ad, wd = a.to(DEV), w.to(DEV)
    _say(f"mid silu norm={norm} {NAME[dout]}")
    if norm:
        nw = (torch.randn(k, generator=torch.Generator().manual_seed(5)) * 0.1).bfloat16().to(DEV)
        run = lambda x: K.gemm_add_rmsnorm_with_kernel(x, x, nw, wd, 1e-6, L.KERNEL_MFMA_STAGED, True, dout)[0]  # noqa: E731
    else:
        run = lambda x: G.gemm_silu_mul_with_kernel(x, wd, L.KERNEL_MFMA_STAGED, dout)  # noqa: E731
    out = run(ad)
    assert L.last_kernel() == "mfma_mid 128x128"
    for r0 in (0, 100, m - 100):
        part = run(ad[r0:r0 + 100])
        torch.cuda.synchronize()
        assert torch.equal(out[r0:r0 + 100], part), f"rows {r0}: {int((out[r0:r0 + 100] != part).sum())} outputs differ"
    if not norm:
        _check_silu_mul(out.cpu(), a, w, dout, rows=np.array([0, 64, 127, 128, m - 1]))
