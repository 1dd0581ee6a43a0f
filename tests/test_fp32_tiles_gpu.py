"""GPU tests of fp32_buffered's tiles by grid size (csrc/gemm_fp32.hip): 16 x 32
(up to 512 of them), 32 x 32, 32 x 64, 64 x 32 and 64 x 64, at the edges of tiles
and of their 64- or 32-wide K-tiles: few K-tiles of each first, then more than are
loaded ahead, so that the loop's steady state runs, with a tail."""
from __future__ import annotations

import importlib

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, LAYOUT, _check_tolerance, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")

SHAPES = [(1, 4, 4), (17, 36, 60), (15, 28, 64), (33, 100, 68), (16, 8196, 132), (50, 1000, 388),
          (33, 8200, 72), (330, 1500, 132), (700, 2052, 68), (2050, 1028, 36)]


# (layout, M, N, K, tile): 7 to 16 K-tiles and a tail.
FORMS = [("nk", 50, 1000, 452, "16x32"), ("kn", 50, 1000, 452, "16x32"), ("nk", 200, 2044, 516, "32x32"),
         ("kn", 200, 2044, 516, "32x32"), ("nk", 700, 2052, 260, "32x64"), ("kn", 700, 2052, 260, "32x64"),
         ("nk", 330, 1500, 260, "64x64"), ("kn", 330, 1500, 452, "64x32"), ("nk", 529, 1092, 196, "64x32"),
         ("nk", 1816, 524, 452, "64x32"), ("kn", 1816, 524, 452, "64x32"), ("nk", 60, 8188, 1100, "64x32"),
         ("nk", 2050, 1028, 260, "64x64"), ("kn", 2050, 1028, 260, "64x64")]


@pytest.mark.parametrize("m,n,k", SHAPES, ids=lambda v: str(v))
@pytest.mark.parametrize("layout", [L.B_NK, L.B_KN], ids=["nk", "kn"])
def test_fp32_tiles(m, n, k, layout):
    _run(m, n, k, layout)


@pytest.mark.parametrize("layout,m,n,k,tile", FORMS, ids=lambda v: str(v))
def test_fp32_forms(layout, m, n, k, tile):
    _run(m, n, k, L.B_NK if layout == "nk" else L.B_KN)
    assert L.last_kernel() == f"fp32_buffered {tile}"


def _run(m, n, k, layout):
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn((m, k), generator=gen)
    b = torch.randn((n, k) if layout == L.B_NK else (k, n), generator=gen) * 0.1
    _say(f"fp32 tiles {LAYOUT[layout]} M={m} N={n} K={k}")
    out = G.gemm_with_kernel(a.to(DEV), b.to(DEV), L.KERNEL_FP32_TILED, torch.float32, layout)
    torch.cuda.synchronize()
    _check_tolerance(out.cpu(), a, b, layout, torch.float32)
