"""GPU tests of fp32_buffered's tiles by grid size (csrc/gemm_fp32.hip): 16 x 32
(up to 512 of them), 32 x 32, 32 x 64 and 64 x 64, at the edges of tiles and of
their 64-wide K-tiles (fewer, as many and more than are loaded ahead)."""
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


@pytest.mark.parametrize("m,n,k", SHAPES, ids=lambda v: str(v))
@pytest.mark.parametrize("layout", [L.B_NK, L.B_KN], ids=["nk", "kn"])
def test_fp32_tiles(m, n, k, layout):
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn((m, k), generator=gen)
    b = torch.randn((n, k) if layout == L.B_NK else (k, n), generator=gen) * 0.1
    _say(f"fp32 tiles {LAYOUT[layout]} M={m} N={n} K={k}")
    out = G.gemm_with_kernel(a.to(DEV), b.to(DEV), L.KERNEL_FP32_TILED, torch.float32, layout)
    torch.cuda.synchronize()
    _check_tolerance(out.cpu(), a, b, layout, torch.float32)
