"""Operands that the kernels read by pointer (dX: the adapter's (dY s) . B and the
dropout mask; the forward: the adapter's own input): a wrong shape, dtype, layout or device raises on the host, before
any library call.  The library is replaced, so no GPU is needed."""
import contextlib

import pytest
import torch

from rocm_qlora import _native as nat
from rocm_qlora import ops

M, N, K, R = 6, 64, 128, 12


class _Launched(Exception):
    pass


@pytest.fixture
def no_library(monkeypatch):
    def require(*tensors):
        devs = {t.device for t in tensors if t is not None}
        if len(devs) != 1:
            raise RuntimeError(f"tensors on different devices: {devs}")
        return devs.pop()

    def call(name, *args):
        raise _Launched(name)

    monkeypatch.setattr(nat, "require_gpu", require)
    monkeypatch.setattr(nat, "call", call)
    monkeypatch.setattr(nat, "stream_handle", lambda dev: 0)
    monkeypatch.setattr(ops, "on", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(ops, "_workspace", lambda *args: None)
    monkeypatch.setattr(ops, "_bytes", lambda fn, dev, *args: 64)


def _nf4(**kw):
    return ops.nf4_linear_dx(torch.zeros(M, N, dtype=torch.bfloat16), torch.zeros(N * K // 2, dtype=torch.uint8),
                             torch.ones(N * K // 64), K, 64, **kw)


def _int8(**kw):
    kw.pop("lora_b", None), kw.pop("scaling", None)
    return ops.int8_linear_dx(torch.zeros(M, N, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.int8),
                              torch.ones(N * K // 64), K, 64, **kw)


def _adapter(**kw):
    return dict(lora_a=torch.zeros(R, K), lora_b=torch.zeros(N, R), scaling=2.0, **kw)


def _g(rows=M, cols=16, dtype=torch.bfloat16):
    return torch.zeros(rows, cols, dtype=dtype)


@pytest.mark.parametrize("fn", [_nf4, _int8])
def test_right_operands_reach_the_library(no_library, fn):
    for kw in (_adapter(lora_g=_g()), _adapter(lora_g=_g(), lora_mask=torch.ones(M, K, dtype=torch.bool), mask_scale=1.25)):
        with pytest.raises(_Launched):
            fn(**kw)


@pytest.mark.parametrize("fn", [_nf4, _int8])
@pytest.mark.parametrize("bad", [_g(cols=R), _g(rows=M - 1), _g(cols=32), _g(dtype=torch.float16), _g(dtype=torch.float32),
                                 _g(rows=16, cols=M).t(), _g(cols=32)[:, ::2], _g(rows=2 * M)[::2], _g().to("meta")],
                         ids=["rank_columns", "short", "wide", "fp16", "fp32", "transposed", "every_other_column",
                              "every_other_row", "device"])
def test_wrong_lora_g_raises(no_library, fn, bad):
    with pytest.raises(RuntimeError):
        fn(**_adapter(lora_g=bad))


@pytest.mark.parametrize("fn", [_nf4, _int8])
def test_lora_g_without_adapters_raises(no_library, fn):
    with pytest.raises(RuntimeError):
        fn(lora_g=_g())


@pytest.mark.parametrize("fn", [_nf4, _int8])
@pytest.mark.parametrize("bad", [torch.ones(M - 1, K, dtype=torch.bool), torch.ones(M, K, dtype=torch.bool, device="meta")],
                         ids=["short", "device"])
def test_wrong_lora_mask_raises(no_library, fn, bad):
    with pytest.raises(RuntimeError):
        fn(**_adapter(lora_g=_g(), lora_mask=bad))


@pytest.mark.parametrize("bad", [torch.zeros(M - 1, K), torch.zeros(2 * M, K), torch.zeros(M, K, device="meta")],
                         ids=["short", "long", "device"])
def test_wrong_lora_x_raises(no_library, bad):
    x, packed, s = torch.zeros(M, K, dtype=torch.bfloat16), torch.zeros(N * K // 2, dtype=torch.uint8), torch.ones(N * K // 64)
    with pytest.raises(_Launched):
        ops.nf4_linear(x, packed, s, N, 64, **_adapter(lora_x=torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        ops.nf4_linear(x, packed, s, N, 64, **_adapter(lora_x=bad))
