"""GPU tests of mfma_staged's 256 x 256 tiles (csrc/gemm_wide.hip): grids that
take them at the edges of tiles, K-tiles and the C tile's store, against the
same rows computed 100 at a time (smaller tiles, which sum K in the same
order, so every bit is equal) and against the oracle."""
from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, NAME, _check_tolerance, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
K = importlib.import_module("inference_systems_amd.kernels.prologue")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _blocks(m):
    """Row ranges on both sides of the tile boundaries and at both ends."""
    return [(0, 100), (200, 300), (m - 356, m - 256), (m - 100, m)]


def _inputs(m, rows, k, dtype):
    gen = torch.Generator().manual_seed(m + rows + k)
    return torch.randn((m, k), generator=gen).to(dtype), (torch.randn((rows, k), generator=gen) * 0.1).to(dtype)


# 160-192 tiles of 256 x 256, and 400 (a round and a part).  N = 3333 and 3334
# store element by element in the last column of tiles (and, with 2-byte outputs,
# in every tile: rows are not 16-byte aligned); K = 256 / 264 / 320 / 328 is 4-6
# K-tiles with tails of 0, 8, 0 and 8.  1301 x 12290 (294 tiles) runs 128-row tiles:
# 256 x 256 would leave most of a second round idle.
@pytest.mark.parametrize("m,n,k,din,dout", [
    (2900, 3333, 264, BF16, BF16), (2900, 3333, 264, BF16, F32), (4096, 2560, 256, BF16, BF16),
    (1301, 12290, 328, F16, F16), (2817, 4096, 320, F16, F32), (2900, 3334, 328, F16, F16),
    (5000, 5000, 328, BF16, BF16)], ids=lambda v: NAME.get(v, v))
def test_wide_tiles(m, n, k, din, dout):
    a, w = _inputs(m, n, k, din)
    ad, wd = a.to(DEV), w.to(DEV)
    _say(f"wide M={m} N={n} K={k} {NAME[din]}->{NAME[dout]}")
    out = G.gemm_with_kernel(ad, wd, L.KERNEL_MFMA_STAGED, dout)
    assert L.last_kernel() == ("mfma_mid 128x256" if n == 12290 else "mfma_wide 256x256")
    for r0, r1 in _blocks(m):
        part = G.gemm_with_kernel(ad[r0:r1], wd, L.KERNEL_MFMA_STAGED, dout)
        torch.cuda.synchronize()
        assert torch.equal(out[r0:r1], part), f"rows {r0}-{r1 - 1}: {int((out[r0:r1] != part).sum())} outputs differ"
    rows = np.array([0, 127, 128, 255, 256, m - 1])
    _check_tolerance(out.cpu(), a, w, L.B_NK, dout, rows=rows)


@pytest.mark.parametrize("dout", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "add-norm"])
def test_wide_tiles_silu(norm, dout):
    """The gate/up pairs (and the row scale of the norm prologue) of the wide
    epilogue: 168 tiles, a ragged last tile in both directions."""
    m, n, k = 2900, 1667, 264
    a, w = _inputs(m, 2 * n, k, BF16)
    gen = torch.Generator().manual_seed(5)
    r, nw = torch.randn((m, k), generator=gen).to(BF16).to(DEV), (torch.randn(k, generator=gen) * 0.1).to(BF16).to(DEV)
    ad, wd = a.to(DEV), w.to(DEV)
    _say(f"wide silu norm={norm} ->{NAME[dout]}")

    def run(r0, r1):
        if norm:
            return K.gemm_add_rmsnorm(ad[r0:r1], r[r0:r1], nw, wd, 1e-6, silu_mul=True, out_dtype=dout)[0]
        return G.gemm_silu_mul_with_kernel(ad[r0:r1], wd, L.KERNEL_MFMA_STAGED, dout)

    out = run(0, m)
    assert L.last_kernel() == "mfma_wide 256x128"
    for r0, r1 in _blocks(m):
        part = run(r0, r1)
        torch.cuda.synchronize()
        assert torch.equal(out[r0:r1], part), f"rows {r0}-{r1 - 1}: {int((out[r0:r1] != part).sum())} outputs differ"
