"""GPU tests of mfma_direct's tiles for rows that are no aligned 16-byte chunks
(csrc/gemm_ragged.hip), against the oracle: every tile choice at its edges, K
and N around chunk and K-tile ends, operands at odd element offsets with odd
leading dimensions, and NaN between the rows, which no load may bring in."""
from __future__ import annotations

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import CODE, DEV, LAYOUT, NAME, _check_tolerance, _say

pytestmark = pytest.mark.gpu

L = PKG._lib
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _framed(x, pad, offset):
    """x in a buffer of its own: row stride cols + pad, first element `offset`
    elements in, NaN everywhere else.  Returns (buffer, address, stride)."""
    rows, cols = x.shape
    ld = cols + pad
    buf = torch.full((offset + rows * ld,), float("nan"), dtype=x.dtype)
    buf[offset:].view(rows, ld)[:, :cols] = x
    buf = buf.to(DEV)
    return buf, buf.data_ptr() + offset * x.element_size(), ld


# Tiles: 32 x 32 (small grids), 16 x 32 (M <= 16, 261 tiles of it), 32 x 64
# (514 tiles of 32 x 32) and 64 x 64 (528 of 64 x 64); K of two chunks and one
# element more, less than three, and around the ends of 64- and 128-element
# K-tiles and of the K-tiles loaded ahead (up to four); up to 16 elements run
# mfma_direct's own kernel.
SHAPES = [(1, 8, 8), (33, 31, 9), (31, 33, 15), (33, 31, 17), (31, 33, 23), (47, 130, 31), (5, 70, 63), (32, 32, 65), (40, 100, 127), (64, 65, 129),
          (70, 33, 257), (17, 50, 391), (3, 9, 520), (16, 8321, 131), (63, 8209, 72 + 1), (1000, 2051, 67)]


@pytest.mark.parametrize("m,n,k", SHAPES, ids=lambda v: str(v))
@pytest.mark.parametrize("layout", [L.B_NK, L.B_KN], ids=["nk", "kn"])
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_ragged_tiles(m, n, k, layout, din, dout):
    gen = torch.Generator().manual_seed(m + n + k)
    a = torch.randn((m, k), generator=gen).to(din)
    b = (torch.randn((n, k) if layout == L.B_NK else (k, n), generator=gen) * 0.1).to(din)
    _say(f"ragged {LAYOUT[layout]} M={m} N={n} K={k} {NAME[din]}->{NAME[dout]}")
    # Odd offsets and strides, and the dense operands one element off alignment.
    for pad_a, pad_b, off in ((3, 5, 7), (0, 0, 1)):
        abuf, ap, lda = _framed(a, pad_a, off)
        bbuf, bp, ldb = _framed(b, pad_b, off)
        ldc = n + 3
        c = torch.full((m, ldc), 7.0, dtype=dout, device=DEV)
        L.gemm_raw(ap, bp, c.data_ptr(), m, n, k, lda, ldb, ldc, layout, CODE[din], CODE[dout],
                   torch.cuda.current_stream().cuda_stream, kernel=L.KERNEL_MFMA_DIRECT)
        assert L.last_kernel().startswith("mfma_direct" if k <= 16 else "mfma_ragged")
        torch.cuda.synchronize()
        _check_tolerance(c[:, :n].cpu(), a, b, layout, dout)
        assert bool((c[:, n:] == 7.0).all()), "a padding column was written"
        del abuf, bbuf
