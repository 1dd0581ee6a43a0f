"""GPU tests of splitk_decode with the rows of A spread over workgroups
(csrc/gemm_decode.hip, launch_rows): row counts on both sides of every block of
8, 16 and 32 rows, ragged N and a partial last line of K.  Every choice adds the
same K partitions in order (16 up to M = 32, 8 above), so a row's bits do not
depend on the rows beside it."""
from __future__ import annotations

import importlib

import pytest
import torch

from conftest import PKG
from test_gemm_gpu import DEV, NAME, _check_tolerance, _say
from test_prologue_gpu import _check_add_norm, _check_add_norm_silu, _norm_inputs, _qgate

pytestmark = pytest.mark.gpu

L = PKG._lib
G = importlib.import_module("inference_systems_amd.kernels.gemm")
K = importlib.import_module("inference_systems_amd.kernels.prologue")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("n,k", [(500, 136), (1001, 1000), (2040, 328)])
@pytest.mark.parametrize("din,dout", [(BF16, BF16), (F16, F32)], ids=["bf16", "f16-f32"])
def test_row_blocks_plain(n, k, din, dout):
    gen = torch.Generator().manual_seed(n + k)
    a = torch.randn((64, k), generator=gen).to(din)
    w = (torch.randn((n, k), generator=gen) * 0.1).to(din)
    ad, wd = a.to(DEV), w.to(DEV)
    alone = torch.cat([G.gemm_with_kernel(ad[i:i + 8], wd, L.KERNEL_SPLITK_DECODE, dout) for i in range(0, 64, 8)])
    torch.cuda.synchronize()
    _check_tolerance(alone.cpu(), a, w, L.B_NK, dout)
    for m in (9, 16, 17, 25, 32, 64, 33, 49):
        _say(f"splitk row blocks M={m} N={n} K={k} {NAME[din]}->{NAME[dout]}")
        out = G.gemm_with_kernel(ad[:m], wd, L.KERNEL_SPLITK_DECODE, dout)
        torch.cuda.synchronize()
        if m == 64:
            _check_tolerance(out.cpu(), a, w, L.B_NK, dout)
            alone = out
        assert torch.equal(out, alone[:m]), f"M={m}: {int((out != alone[:m]).sum())} outputs differ"


@pytest.mark.parametrize("m", [9, 17, 31])
@pytest.mark.parametrize("n", [500, 1001, 2200])
def test_row_blocks_gate(m, n):
    """The gate fused into blocks of 8 rows (the default while the workgroups
    fit the CUs), against the gate kernel followed by the GEMM: bit-exact."""
    gen = torch.Generator().manual_seed(m + n)
    a = torch.randn((m, 5, 64), generator=gen).bfloat16().to(DEV)
    gate = _qgate(m, 5, 64, BF16, gen)[0].to(DEV).chunk(2, -1)[1]
    w = (torch.randn((n, 320), generator=gen) * 0.05).bfloat16().to(DEV)
    _say(f"gate row blocks M={m} N={n}")
    got = K.gemm_gated(a, gate, w)
    want = G.gemm_with_kernel(K.sigmoid_gate(a, gate), w, L.KERNEL_SPLITK_DECODE)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


# n: 16-row blocks of W with 8 rows of A (500), 16 (2000), and with SiLU pairs 8
# rows (500), 16 rows on 16 pairs (1500) and 16 rows on 32 pairs (3000).
@pytest.mark.parametrize("silu,n", [(False, 500), (False, 2000), (True, 500), (True, 1500), (True, 3000)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("m", [9, 17, 25, 32])
def test_row_blocks_add_norm(silu, n, m):
    k = 200
    gen = torch.Generator().manual_seed(m + n + silu)
    h, r, nw, w = _norm_inputs(m, 2 * n if silu else n, k, BF16, gen)
    _say(f"add_rmsnorm row blocks M={m} N={n} silu={silu}")
    out, res = K.gemm_add_rmsnorm(h.to(DEV), r.to(DEV), nw.to(DEV), w.to(DEV), 1e-6, silu_mul=silu)
    torch.cuda.synchronize()
    (_check_add_norm_silu if silu else _check_add_norm)(out, res, h, r, nw, w, 1e-6, BF16, BF16)


def test_gate_kernel_group_placement():
    """The stand-alone gate on a head size that is no power of two and more
    chunks than one block takes, against the two roundings in torch."""
    m, heads, hd = 37, 7, 40
    gen = torch.Generator().manual_seed(3)
    a = torch.randn((m, heads, hd), generator=gen).bfloat16()
    gate = torch.randn((m, heads, 2 * hd), generator=gen).bfloat16().chunk(2, -1)[1]
    got = K.sigmoid_gate(a.to(DEV), torch.cat([gate, gate], -1).to(DEV).chunk(2, -1)[1]).cpu()
    sg = torch.sigmoid(gate.double())
    want = (a.double() * sg).reshape(m, -1)
    # two roundings to bf16, of the sigmoid and of the product: 2^-8 each
    assert bool(((got.double() - want).abs() <= want.abs() * (2 ** -7 + 2 ** -12)).all())


@pytest.mark.parametrize("k", [1024, 4096])
def test_gate_without_workspace(k):
    """Up to 8 rows the C ABI takes no workspace: the fused gate runs, at any K,
    with the bits of the path that has one."""
    m, n = 8, 520
    gen = torch.Generator().manual_seed(k)
    a = torch.randn((m, k // 64, 64), generator=gen).bfloat16().to(DEV)
    gate = torch.randn((m, k // 64, 64), generator=gen).bfloat16().to(DEV)
    w = (torch.randn((n, k), generator=gen) * 0.05).bfloat16().to(DEV)
    out = torch.empty((m, n), dtype=BF16, device=DEV)
    L.gated_raw(a.data_ptr(), gate.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, k, k, 64, 64, k, n, L.BF16, L.BF16,
                None, 0, torch.cuda.current_stream().cuda_stream)
    want = K.gemm_gated(a, gate, w)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
