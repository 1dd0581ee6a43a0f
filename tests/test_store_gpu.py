"""GPU tests of the C tile's store to rows that are not 16-byte aligned
(store_unaligned, csrc/gemm_common.hpp) from every family of MFMA tiles: words
where rows are 4-byte aligned, with an odd last column, and elements otherwise;
the dense, aligned product bit for bit, nothing written beside it."""
from __future__ import annotations

import importlib

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import CODE, DEV, NAME, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


FORMS = {(70, 136): "narrow 32x32", (1100, 136): "staged 64x64", (1100, 264): "staged 64x64",
         (2200, 264): "mid 128x128", (2300, 264): "mid 128x256", (5000, 264): "wide 256x256"}


@pytest.mark.parametrize("m,k", FORMS, ids=lambda v: str(v))
@pytest.mark.parametrize("n", [1032, 1031], ids=["even", "odd"])
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_unaligned_rows(m, n, k, din, dout):
    n *= 2 if m >= 2300 else 1
    gen = torch.Generator().manual_seed(m + n)
    a = torch.randn((m, k), generator=gen).to(din).to(DEV)
    w = torch.randn((n, k), generator=gen).to(din).to(DEV)
    _say(f"unaligned store M={m} N={n} K={k} {NAME[dout]}")
    full = torch.empty((m, (n + 7) // 8 * 8), dtype=dout, device=DEV)

    def run(c, ldc):
        L.gemm_raw(a.data_ptr(), w.data_ptr(), c.data_ptr(), m, n, k, k, k, ldc, L.B_NK, CODE[din], CODE[dout],
                   torch.cuda.current_stream().cuda_stream, kernel=L.KERNEL_MFMA_STAGED)

    run(full, full.shape[1])
    assert L.last_kernel() == f"mfma_{FORMS[m, k]}"
    for ldc, first in ((n + 1, 0), (n + 2, 0), (n + 4, 1), (n + 4, 2)):
        buf = torch.full((first + m * ldc,), 7.0, dtype=dout, device=DEV)
        c = buf[first:].view(m, ldc)
        run(c, ldc)
        torch.cuda.synchronize()
        assert torch.equal(c[:, :n], full[:, :n]), f"ldc={ldc} first={first}"
        assert bool((c[:, n:] == 7.0).all()) and bool((buf[:first] == 7.0).all()), "wrote beside C"
