"""The fused ops registered from C++ (csrc/torch_ops.cpp): schemas and messages
those of the ctypes registration, results its bits, and no backward."""
from __future__ import annotations

import importlib
import json
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from conftest import PKG

G = importlib.import_module("inference_systems_amd.kernels.gemm")
K = importlib.import_module("inference_systems_amd.kernels.prologue")
L = PKG._lib
DEV = "cuda"
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

_PROBE = r"""
import json, sys
sys.path.insert(0, {root!r})
import torch
import __graft_entry__ as g
g.load_package()
ops = torch.ops.nanovllm
a = torch.randn(4, 64).bfloat16()
out = []
for name, args in (("gemm_silu_mul", (a, a)), ("gemm_argmax", (a, a)), ("gemm_sample", (a, a, torch.zeros(4), 1, 2)),
                   ("gemm_gated", (a, a, a)), ("gemm_add_rmsnorm", (a, a, a[0], a, 1e-6))):
    op = getattr(ops, name)
    try:
        op(*args)
    except RuntimeError as exc:
        out.append([str(op.default._schema), str(exc).splitlines()[0]])
print(json.dumps(out))
"""


def test_registrations_share_schemas_and_messages():
    root = str(Path(__file__).resolve().parents[1])
    got = {}
    for choice in ("torch_library", "custom_op"):
        env = dict(os.environ, **{G.OPS_ENV: choice})
        env.pop("NANOVLLM_GEMM_LIB", None)
        proc = subprocess.run([sys.executable, "-c", _PROBE.format(root=root)], env=env, capture_output=True, text=True,
                              timeout=300)
        assert proc.returncode == 0, proc.stderr
        got[choice] = json.loads(proc.stdout.strip().splitlines()[-1])
    assert len(got["torch_library"]) == 5
    assert got["torch_library"] == got["custom_op"]


def test_hip_backend_refuses_meta_tensors():
    """A fake implementation must not stand in for operands off the GPU."""
    a, w = torch.empty((4, 64), device="meta", dtype=BF16), torch.empty((8, 64), device="meta", dtype=BF16)
    with pytest.raises(RuntimeError, match="HIP GEMM backend is unavailable: a and w must be CUDA"):
        G.linear(a, w, backend="hip")
    with pytest.raises(RuntimeError, match="HIP GEMM backend is unavailable: a, gate and w must be CUDA"):
        K.gated_linear(a, a, w, backend="hip")


def _randn(*shape, dtype=BF16):
    gen = torch.Generator().manual_seed(sum(shape))
    return (torch.randn(shape, generator=gen) * 0.2).to(dtype).to(DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 20, 100])
def test_same_bits_as_ctypes(m):
    """Every fused op against its ctypes launch, default and fp32 outputs."""
    a, w, gu = _randn(m, 128), _randn(200, 128), _randn(400, 128)
    gate = _randn(m, 2, 128).chunk(2, -1)[1]
    nw, t = _randn(128), torch.linspace(0, 1.5, m, device=DEV)
    ops = torch.ops.nanovllm
    for od in (None, F32):
        assert torch.equal(ops.gemm_silu_mul(a, gu, od), G._launch_silu_mul(a, gu, od))
        assert torch.equal(ops.gemm_gated(a.view(m, 2, 64), gate, w, od), K._launch_gated(a.view(m, 2, 64), gate, w, od))
        for silu in (False, True):
            for x, y in zip(ops.gemm_add_rmsnorm(a, a, nw, gu, 1e-6, silu, od),
                            K._launch_add_rmsnorm(a, a, nw, gu, 1e-6, silu, od)):
                assert torch.equal(x, y)
        for x, y in zip(ops.gemm_argmax(a, w, od), G._launch_argmax(a, w, od)):
            assert torch.equal(x, y)
        # seeds and offsets of all 64 bits
        for seed in (3, -5):
            for x, y in zip(ops.gemm_sample(a, w, t, seed, -2, od), G._launch_sample(a, w, t, seed, -2, od)):
                assert torch.equal(x, y)


@pytest.mark.gpu
def test_messages_on_gpu():
    """Each violation raises what the Python contract says, from the op and
    from the hip backend."""
    a, w, nw = _randn(4, 64), _randn(8, 64), _randn(64)
    odd = _randn(4 * 64 + 8)[1:257].view(4, 64)   # not 16-byte aligned
    ops = torch.ops.nanovllm
    silu = [(a, w.half()), (a, _randn(9, 64)), (a.float(), w.float()), (_randn(4, 60), _randn(8, 60)), (odd, w),
            (a, _randn(64, 8).T)]
    for x, y in silu:
        why = G.silu_mul_contract_reason(x, y)
        assert why is not None
        with pytest.raises(RuntimeError) as err:
            ops.gemm_silu_mul(x, y)
        assert str(err.value).splitlines()[0] == f"nanovllm::gemm_silu_mul: {why}"
        with pytest.raises(RuntimeError) as err:
            G.silu_mul_linear(x, y, backend="hip")
        assert str(err.value) == f"HIP GEMM backend is unavailable: {why}"
    t = torch.zeros(4, device=DEV)
    head = [(a.float(), w.float(), t), (_randn(4, 60), _randn(8, 60), t), (odd, w, t), (a, w, t.double()),
            (a, w, torch.zeros(4)), (a, w, torch.zeros(3, device=DEV)), (a, w, torch.zeros((4, 1), device=DEV)),
            (a, w, torch.zeros(8, device=DEV)[::2]), (a, _randn(0, 64), t)]
    for x, y, temps in head:
        why = G.sample_contract_reason(x, y, temps)
        assert why is not None
        with pytest.raises(RuntimeError) as err:
            ops.gemm_sample(x, y, temps, 1, 2)
        assert str(err.value).splitlines()[0] == f"nanovllm::gemm_sample: {why}"
    with pytest.raises(RuntimeError, match="logits_dtype must be None, torch.bfloat16 or torch.float32, got torch.float16"):
        ops.gemm_argmax(a, w, F16)
    g3 = _randn(4, 2, 64)
    gated = [(a, a, w, F16), (a.float(), a.float(), w.float(), None), (a, a.half(), w, None), (a, a, _randn(8, 32), None),
             (a, _randn(4, 32), w, None), (a, g3, w, None), (a, _randn(4, 128)[:, ::2], w, None),
             (a, _randn(4, 2, 36)[:, :, :32], w, None), (a, odd, w, None), (a, nw, w, None), (_randn(64), a, w, None)]
    for x, g, y, od in gated:
        why = K.gated_contract_reason(x, g, y, od)
        assert why is not None
        with pytest.raises(RuntimeError) as err:
            ops.gemm_gated(x, g, y, od)
        assert str(err.value).splitlines()[0] == f"nanovllm::gemm_gated: {why}"
    with pytest.raises(IndexError):
        ops.gemm_gated(a[:0], a[:0], w)
    norm = [(a.half(), a.half(), nw.half(), w.half(), False, None), (a, a, nw, w.half(), False, None), (a, a, nw, w, False, F16),
            (a, _randn(3, 64), nw, w, False, None), (a, a, _randn(32), w, False, None), (a, a, nw, _randn(8, 32), False, None),
            (a, a, nw, _randn(9, 64), True, None), (a, a, nw, _randn(0, 64), False, None),
            (a, _randn(64, 4).T, nw, w, False, None), (_randn(4, 60), _randn(4, 60), _randn(60), _randn(8, 60), False, None),
            (a, odd, nw, w, False, None)]
    for x, r, n, y, s, od in norm:
        why = K.add_rmsnorm_contract_reason(x, r, n, y, s, od)
        assert why is not None
        with pytest.raises(RuntimeError) as err:
            ops.gemm_add_rmsnorm(x, r, n, y, 1e-6, s, od)
        assert str(err.value).splitlines()[0] == f"nanovllm::gemm_add_rmsnorm: {why}"


@pytest.mark.gpu
def test_backward_is_refused():
    a = _randn(4, 64).requires_grad_()
    w = _randn(8, 64)
    for y in (torch.ops.nanovllm.gemm_silu_mul(a, w), torch.ops.nanovllm.gemm_gated(a, a.detach(), w),
              torch.ops.nanovllm.gemm_add_rmsnorm(a, a.detach(), w[0], w, 1e-6)[0]):
        with pytest.raises(RuntimeError):
            y.float().sum().backward()
