"""The adapters' gradients where the HIP kernels cannot run: batched output
gradients (torch.autograd.grad(is_grads_batched=True), tensors without storage)
and forward-mode AD take the torch expressions, on any device; and calls inside
torch.jit.trace keep their autograd functions, without which the trace would hold
an output allocation and nothing that fills it."""
import pytest
import torch
from torch.autograd import forward_ad

from rocm_qlora import ops
from rocm_qlora.kernels import dequant_matmul as dm


class _Adapter(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, a, b, s):
        ctx.save_for_backward(x, a, b)
        ctx.s = s
        return x @ a.T @ b.T * s

    @staticmethod
    def backward(ctx, dy):
        x, a, b = ctx.saved_tensors
        da, db, _ = dm._lora_backward(dy, x, a, b, ctx.s, True, True, False)
        return None, da, db, None


@pytest.fixture
def kernels_refused(monkeypatch):
    def refuse(*a, **k):
        raise AssertionError("the gradient kernels were called")
    monkeypatch.setattr(ops, "lora_grads", refuse)


def _inputs():
    g = torch.Generator().manual_seed(0)
    x, a, b = (torch.randn(s, generator=g).bfloat16() for s in ((5, 64), (8, 64), (32, 8)))
    return x, a.requires_grad_(), b.requires_grad_(), torch.randn((3, 5, 32), generator=g).bfloat16()


def test_batched_gradients(kernels_refused):
    x, a, b, dys = _inputs()
    got = torch.autograd.grad(_Adapter.apply(x, a, b, 2.0), (a, b), dys, is_grads_batched=True)
    for i, dy in enumerate(dys):
        ref = torch.autograd.grad(x @ a.T @ b.T * 2.0, (a, b), dy)
        for p, q in zip(got, ref):  # one rounding per intermediate: 3 of 2^-9 in the 2-norm
            assert (p[i] - q).float().norm() <= 3 * 2.0 ** -9 * q.float().norm()


def test_forward_mode_gradients(kernels_refused):
    x, a, b, dys = _inputs()
    with forward_ad.dual_level(), torch.no_grad():
        dm._lora_backward(dys[0], x, a, b, 2.0, True, True, False)


def test_calls_inside_jit_trace_keep_their_autograd_function():
    x, a = torch.zeros(5, 64).bfloat16(), torch.zeros(8, 64)
    seen = []

    def f(t):
        seen.append((dm._nothing_recorded(t), dm.native_adapter(t, a)))
        return t + 1

    with torch.no_grad():
        f(x)
        torch.jit.trace(f, (x,), check_trace=False)
    assert seen == [(True, True), (False, False)]
