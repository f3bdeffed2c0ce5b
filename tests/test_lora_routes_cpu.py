"""The adapters' gradients where the HIP kernels cannot run: batched output
gradients (torch.autograd.grad(is_grads_batched=True), tensors without storage)
and forward-mode AD take the torch expressions, on any device; and calls inside
torch.jit.trace keep their autograd functions, without which the trace would hold
an output allocation and nothing that fills it."""
import types

import pytest
import torch
import torch.nn as nn
from torch.autograd import forward_ad

from rocm_qlora import LoRALinear, QuantLinear, ops
from rocm_qlora.fp8 import fp8_linear
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


def _patch_forward(drop):
    forward = drop.forward
    drop.forward = lambda x: forward(x)


class _MyDropout(nn.Dropout):
    pass


# what makes a call of the adapter's dropout module more than its probability
DROPOUTS = {
    "subclass": lambda: _MyDropout(0.1),
    "in_place": lambda: nn.Dropout(0.1, inplace=True),
    "forward_hook": lambda: _with(nn.Dropout(0.1), lambda d: d.register_forward_hook(lambda m, i, o: None)),
    "forward_pre_hook": lambda: _with(nn.Identity(), lambda d: d.register_forward_pre_hook(lambda m, i: None)),
    "backward_hook": lambda: _with(nn.Dropout(0.1), lambda d: d.register_full_backward_hook(lambda m, i, o: None)),
    "backward_pre_hook": lambda: _with(nn.Dropout(0.1), lambda d: d.register_full_backward_pre_hook(lambda m, o: None)),
    "replaced_forward": lambda: _with(nn.Dropout(0.1), _patch_forward),
    "global_hook": lambda: nn.Dropout(0.1),
    "plain": lambda: nn.Dropout(0.1),
    "none": lambda: nn.Identity(),
}


def _with(drop, change):
    change(drop)
    return drop


@pytest.mark.parametrize("kind", DROPOUTS)
def test_fp8_layer_calls_a_dropout_module_that_is_more_than_its_probability(monkeypatch, kind):
    layer = LoRALinear(QuantLinear(64, 32, bits=4, bias=False), r=8, lora_alpha=16)
    layer.lora_dropout = DROPOUTS[kind]()
    wrapper = fp8_linear.FP8LinearWrapper(layer)
    wrapper.backend = "native"
    wrapper._weight = lambda dtype: None
    routes = []
    monkeypatch.setattr(dm, "native_adapter", lambda x, a: True)
    monkeypatch.setattr(dm, "base_lora_linear", lambda *a: routes.append("kernels"))
    monkeypatch.setattr(fp8_linear, "_FP8LinearFunc",
                        types.SimpleNamespace(apply=lambda x, *a: (routes.append("module"), torch.zeros(x.shape[0], 32))[1]))
    hook = nn.modules.module.register_module_forward_hook(lambda m, i, o: None) if kind == "global_hook" else None
    try:
        wrapper(torch.randn(5, 64))
    finally:
        if hook is not None:
            hook.remove()
    assert routes == (["kernels"] if kind in ("plain", "none") else ["module"])
