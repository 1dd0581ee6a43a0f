"""GPU tests of mfma_staged's small tiles (csrc/gemm_narrow.hip): every tile
choice at the edges of tiles, K-tiles and chunks, against the oracle and, bit
for bit, against the same rows inside a launch of more rows, which takes larger
tiles and sums K in the same order."""
from __future__ import annotations

import importlib

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, NAME, _check_silu_mul, _check_tolerance, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
K = importlib.import_module("inference_systems_amd.kernels.prologue")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

# (M, N, K, M of the larger launch).  32 x 32 on K-tiles of 128 (one chunk; a
# K-tile less, more than and of a whole number of chunks; more K-tiles than
# stages) and of 256, 32 x 64, 64 x 64.
NK = [(1, 8, 8, 9000), (33, 100, 120, 4400), (31, 1000, 136, 4400), (40, 96, 1000, 4400), (65, 333, 1544, 4400),
      (100, 40, 2048, 4400), (90, 4104, 136, 1100), (321, 1001, 648, 4400), (500, 1029, 264, 4400),
      (190, 4100, 72, 1500)]
KN = [(33, 104, 120, 4400), (90, 4104, 136, 1100), (321, 1000, 648, 4400), (190, 4104, 72, 1500)]

# The shapes above whose K is too short for a tile of that size run
# mfma_staged's; these run the tiles they name (K of whole K-tiles of 128, and
# with tails of one chunk, of half a K-tile and more).
FORMS = [("NK", 40, 96, 72, 4400, "32x32"), ("NK", 65, 333, 1800, 4400, "32x32"),
         ("NK", 90, 4104, 584, 1100, "32x64"), ("NK", 321, 1001, 648, 4400, "32x64"),
         ("NK", 320, 1472, 384, 4400, "32x64"), ("NK", 500, 1029, 1800, 4400, "64x64"),
         ("NK", 190, 4100, 512, 1500, "64x64"), ("NK", 449, 1500, 576, 3000, "64x64"),
         ("KN", 33, 104, 776, 4400, "32x64"), ("KN", 90, 4104, 840, 1100, "32x64"), ("KN", 200, 512, 512, 4400, "32x64"),
         ("KN", 190, 4104, 2056, 1500, "64x64"), ("KN", 449, 1472, 1088, 3000, "64x64")]


def _run(m, n, k, mm, din, dout, layout, tile=None):
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn((mm, k), generator=gen).to(din)
    b = (torch.randn((n, k) if layout == L.B_NK else (k, n), generator=gen) * 0.1).to(din)
    ad, bd = a.to(DEV), b.to(DEV)
    _say(f"narrow M={m} N={n} K={k} layout={layout} {NAME[din]}->{NAME[dout]}")
    out = G.gemm_with_kernel(ad[:m], bd, L.KERNEL_MFMA_STAGED, dout, layout)
    if tile is not None:
        assert L.last_kernel() == f"mfma_narrow {tile}"
    big = G.gemm_with_kernel(ad, bd, L.KERNEL_MFMA_STAGED, dout, layout)
    assert tile is None or not L.last_kernel().startswith("mfma_narrow")
    torch.cuda.synchronize()
    assert torch.equal(out, big[:m]), f"{int((out != big[:m]).sum())} outputs differ"
    _check_tolerance(out.cpu(), a[:m], b, layout, dout)


@pytest.mark.parametrize("m,n,k,mm", NK, ids=lambda v: str(v))
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_narrow_nk(m, n, k, mm, din, dout):
    _run(m, n, k, mm, din, dout, L.B_NK)


@pytest.mark.parametrize("m,n,k,mm", KN, ids=lambda v: str(v))
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_narrow_kn(m, n, k, mm, din, dout):
    _run(m, n, k, mm, din, dout, L.B_KN)


@pytest.mark.parametrize("layout,m,n,k,mm,tile", FORMS, ids=lambda v: str(v))
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_narrow_forms(layout, m, n, k, mm, tile, din, dout):
    _run(m, n, k, mm, din, dout, L.B_NK if layout == "NK" else L.B_KN, tile)


# Rows x outputs: 32 x 32, 64 x 32 on 8 waves, 64 x 32 two to a CU, and
# mfma_staged's 64 x 64 where rows of that grid are not whole 128-byte lines.
@pytest.mark.parametrize("m,n,k,tile", [
    (40, 1000, 136, "narrow 32x32"), (33, 8, 520, "narrow 32x32"), (70, 3000, 72, "narrow 64x32"),
    (200, 3333, 320, "narrow 64x32"), (200, 3333, 264, "staged 64x64")], ids=lambda v: str(v))
@pytest.mark.parametrize("norm", [False, True], ids=["plain", "add-norm"])
def test_narrow_silu(m, n, k, tile, norm):
    mm = 3000
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn((mm, k), generator=gen).bfloat16()
    w = (torch.randn((2 * n, k), generator=gen) * 0.1).bfloat16()
    ad, wd = a.to(DEV), w.to(DEV)
    _say(f"narrow silu M={m} N={n} K={k} norm={norm}")
    if norm:
        nw = (torch.randn(k, generator=gen) * 0.1).bfloat16().to(DEV)
        run = lambda x: K.gemm_add_rmsnorm_with_kernel(x, x, nw, wd, 1e-6, L.KERNEL_MFMA_STAGED, silu_mul=True)[0]  # noqa: E731
    else:
        run = lambda x: G.gemm_silu_mul_with_kernel(x, wd, L.KERNEL_MFMA_STAGED)  # noqa: E731
    out = run(ad[:m])
    assert L.last_kernel() == f"mfma_{tile}"
    big = run(ad)
    torch.cuda.synchronize()
    assert torch.equal(out, big[:m]), f"{int((out != big[:m]).sum())} outputs differ"
    if not norm:
        _check_silu_mul(out.cpu(), a[:m], w, BF16)
