"""GPU tests of which kernel and tile a problem runs on: shapes on both sides of
the dispatch rules (nanovllm_gemm_last_kernel names what the call launched).
Every form of a kernel id gives the same bits, so only the names, and the time,
tell a wrong rule."""
from __future__ import annotations

import importlib

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def ran(m, n, k, dtype=BF16, out=None, kn=False, silu=False):
    a = torch.zeros((m, k), dtype=dtype, device=DEV)
    w = torch.zeros((k, n) if kn else (2 * n if silu else n, k), dtype=dtype, device=DEV)
    _say(f"last kernel {m}x{n}x{k} kn={kn} silu={silu}")
    if silu:
        G.gemm_silu_mul(a, w, out)
    else:
        (G.gemm_kn if kn else G.gemm)(a, w, out)
    torch.cuda.synchronize()
    return L.last_kernel()


@pytest.mark.parametrize("m,n,k,dtype,want", [
    (1, 512, 256, BF16, "gemv_decode 1x"), (4, 512, 256, BF16, "splitk_decode 8x16"),
    (32, 8192, 256, BF16, "splitk_decode 32x32"), (200, 1024, 512, BF16, "mfma_narrow 32x32"),
    (2048, 4096, 1024, BF16, "mfma_mid 128x256"), (4096, 1024, 1024, F16, "mfma_mid 128x128"),
    (4096, 4096, 512, BF16, "mfma_wide 256x256"), (2048, 4096, 128, BF16, "mfma_staged 128x256"),
    (100, 100, 101, BF16, "mfma_ragged 32x32"), (5, 5, 5, BF16, "mfma_direct 64x64"),
    (100, 128, 128, F32, "fp32_buffered 16x32"), (100, 128, 127, F32, "fp32_tiled 64x64"),
])
def test_kernel_families(m, n, k, dtype, want):
    assert ran(m, n, k, dtype).startswith(want)


@pytest.mark.parametrize("m,n,k,kn,want", [
    # one round of 32 x 32 tiles
    (128, 512, 64, False, "mfma_staged 64x64"), (128, 512, 72, False, "mfma_narrow 32x32"),
    # of 32 x 64: rows of whole 128-byte lines, then not
    (320, 1536, 320, False, "mfma_staged 64x64"), (320, 1536, 384, False, "mfma_narrow 32x64"),
    (320, 1536, 568, False, "mfma_staged 64x64"), (320, 1536, 584, False, "mfma_narrow 32x64"),
    # of 64 x 64
    (700, 1024, 448, False, "mfma_staged 64x64"), (700, 1024, 512, False, "mfma_narrow 64x64"),
    (700, 1024, 1784, False, "mfma_staged 64x64"), (700, 1024, 1800, False, "mfma_narrow 64x64"),
    # more than one round
    (1024, 2048, 512, False, "mfma_staged 64x64"),
    # B[K,N]
    (200, 512, 448, True, "mfma_staged 64x64"), (200, 512, 512, True, "mfma_narrow 32x64"),
    (200, 520, 760, True, "mfma_staged 64x64"), (200, 520, 768, True, "mfma_narrow 32x64"),
    (700, 1024, 960, True, "mfma_staged 64x64"), (700, 1024, 1024, True, "mfma_narrow 64x64"),
    (700, 1000, 2040, True, "mfma_staged 64x64"), (700, 1000, 2048, True, "mfma_narrow 64x64"),
])
def test_small_grids(m, n, k, kn, want):
    """A short K stays on the 64 x 64 tiles with 64-element K-tiles."""
    assert ran(m, n, k, kn=kn) == want


@pytest.mark.parametrize("m,n,k,silu,want", [
    # one part of a round, and one full round and a part: by the model's margin at a short K
    (4096, 2560, 256, False, "mfma_wide 256x256"), (6300, 3648, 256, False, "mfma_mid 128x256"),
    (4757, 2112, 256, True, "mfma_mid 128x128"), (3010, 2688, 320, True, "mfma_wide 256x128"),
    (5321, 6312, 480, False, "mfma_mid 128x256"),
    (5321, 6312, 1024, False, "mfma_wide 256x256"),
])
def test_large_grids(m, n, k, silu, want):
    assert ran(m, n, k, silu=silu) == want


@pytest.mark.parametrize("m,n,k,want", [
    (200, 1200, 264, "mfma_narrow 64x32"), (100, 1000, 264, "mfma_narrow 32x32"),
    # two rounds of 64 x 32 outputs: whole 128-byte lines, not, a very long K, and
    # more than 128 tiles of 128 x 128
    (729, 1216, 1024, "mfma_narrow 64x32"), (729, 1216, 992, "mfma_staged 64x64"),
    (200, 3584, 3072, "mfma_narrow 64x32"), (200, 3584, 3136, "mfma_staged 64x64"),
    (440, 2080, 992, "mfma_narrow 64x32"),
])
def test_small_silu_grids(m, n, k, want):
    assert ran(m, n, k, silu=True) == want


@pytest.mark.parametrize("m,n,k,kn,want", [
    (100, 100, 15, False, "mfma_direct 64x64"), (100, 100, 17, False, "mfma_ragged 32x32"),
    (1500, 1001, 31, True, "mfma_direct 64x64"), (1500, 1001, 33, True, "mfma_ragged 32x64"),
    (1500, 1001, 33, False, "mfma_ragged 32x64"), (100, 7, 65, True, "mfma_direct 64x64"),
    # B[K,N] behind rows of A that are aligned chunks: 35, 340, 400 and 768 tiles
    # of 64 x 64
    (300, 401, 64, True, "mfma_direct 64x64"), (300, 401, 72, True, "mfma_ragged 32x32"),
    (1270, 1051, 64, True, "mfma_direct 64x64"), (1270, 1051, 72, True, "mfma_ragged 32x64"),
    (1270, 1251, 256, True, "mfma_direct 64x64"), (1270, 1251, 264, True, "mfma_ragged 32x64"),
    (2048, 1501, 80, True, "mfma_direct 64x64"), (2048, 1501, 88, True, "mfma_ragged 64x64"),
])
def test_ragged_grids(m, n, k, kn, want):
    assert ran(m, n, k, kn=kn) == want


@pytest.mark.parametrize("m,n,k,kn,want", [
    (16, 4096, 256, False, "16x32"), (200, 2044, 260, False, "32x32"), (200, 2044, 260, True, "32x32"),
    # B of more and of less than 32 MiB, in one round of 64 x 32 tiles or more
    (56, 5316, 1580, False, "64x32"), (56, 5316, 1576, False, "32x32"), (69, 5016, 1720, True, "32x32"),
    (700, 2052, 260, False, "32x64"), (700, 2052, 260, True, "32x64"),
    (330, 1500, 260, False, "64x64"), (330, 1500, 260, True, "64x32"), (529, 1088, 260, False, "64x64"), (529, 1088, 260, True, "64x32"),
    (529, 1088, 196, False, "64x32"), (1816, 524, 260, True, "64x32"), (1816, 524, 260, False, "64x32"),
    (2050, 1028, 260, False, "64x64"),
])
def test_fp32_grids(m, n, k, kn, want):
    assert ran(m, n, k, F32, kn=kn) == f"fp32_buffered {want}"
