"""Fused dequantize + matmul for NF4 and INT8 weights, with autograd
(kernels/dequant_matmul.py:214-376 of the reference).

Forward runs the HIP kernels of this package: a weight-streaming GEMV for up
to 16 activation rows, the MFMA GEMM above that, both with bias and the LoRA
term fused.  Backward returns dX only, as the reference does
(dequant_matmul.py:338-351), plus dA / dB when LoRA adapters are passed:
dX = dY . W_deq (+ ((dY * s) . B) . A) by the NF4 dX kernel.

Every shape, block size and activation dtype (fp32 included) runs on the
library's HIP kernels: shapes the specialized kernels do not take (K not a
multiple of 64, block sizes that are not powers of two >= 64 dividing K,
unaligned rows) run on its generic kernels, which decode the weight inside
the multiply with the same roundings as the reference's
dequantize-then-F.linear path.  INT8 backward is dX = dY . W_deq on those
kernels too.  Tensors on the CPU raise; there is no CPU or library path.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch
from torch.autograd import forward_ad

from rocm_qlora import _native as nat
from rocm_qlora import ops
from rocm_qlora import torch_ops

# activation dtypes of the HIP linear kernels
_KERNEL_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


@dataclass
class NF4Weight:
    """An NF4 weight as QuantLinear stores it: flat packed codes (byte j =
    element 2j low nibble, 2j+1 high nibble) and one absmax per block, or,
    with double quantization, c2 codes plus c2_scales per blocksize_2 blocks."""
    packed: torch.Tensor
    scales: Optional[torch.Tensor]
    N: int
    K: int
    block_size: int = 64
    c2: Optional[torch.Tensor] = None
    c2_scales: Optional[torch.Tensor] = None
    blocksize_2: int = 256
    use_fp8_c2: bool = True

    def kernel_ok(self, dtype: torch.dtype) -> bool:
        """The HIP kernels take this activation dtype (any shape)."""
        return dtype in _KERNEL_DTYPES

    def dq_kwargs(self) -> dict:
        if self.c2 is None:
            return {}
        return dict(c2=self.c2, c2_scales=self.c2_scales, blocksize_2=self.blocksize_2,
                    use_fp8_c2=self.use_fp8_c2)

    def dense(self, dtype: torch.dtype) -> torch.Tensor:
        """[N, K] dequantized weight in `dtype` (dequantize_int4 /
        double_dequantize, then `[:N*K].reshape(N, K).to(dtype)`,
        quant_linear.py:168-193), by the HIP codec kernels."""
        from rocm_qlora.quantization.quant_ops import nf4_dequantize_to
        from rocm_qlora.quantization.double_quant import dq_dequantize_to
        n = self.N * self.K
        if self.c2 is not None:
            w = dq_dequantize_to(self.packed, self.c2, self.c2_scales, self.block_size, self.blocksize_2,
                                 self.use_fp8_c2, dtype, n)
        else:
            w = nf4_dequantize_to(self.packed, self.scales, self.block_size, dtype, n)
        return w.view(self.N, self.K)


@dataclass
class Int8Weight:
    """An int8 weight: per-row scales (block_size 0, the row-absmax recipe,
    q [N, K] with [N] scales) or blockwise scales over the flat weight."""
    q: torch.Tensor
    scales: torch.Tensor
    N: int
    K: int
    block_size: int = 64

    def kernel_ok(self, dtype: torch.dtype) -> bool:
        """The HIP kernels take this activation dtype (any shape)."""
        return dtype in _KERNEL_DTYPES

    def dense(self, dtype: torch.dtype) -> torch.Tensor:
        """[N, K] dequantized weight (dequantize_int8, quant_ops.py:55-78), cast."""
        from rocm_qlora.quantization.quant_ops import dequantize_int8
        n = self.N * self.K
        if self.block_size == 0:
            w = dequantize_int8(self.q.reshape(self.N, self.K), self.scales.reshape(-1))
        else:
            w = dequantize_int8(self.q.reshape(-1), self.scales.reshape(-1), self.block_size)
        return w.reshape(-1)[:n].view(self.N, self.K).to(dtype)


_functorch_active = getattr(torch._C, "_are_functorch_transforms_active", lambda: True)


def _plain_eager() -> bool:
    """Whether the call runs as it stands: no tracing (torch.compile,
    torch.jit.trace), functorch transform or forward-mode AD active."""
    return not torch_ops.compiling() and not torch._C._is_tracing() and not _functorch_active() and \
        forward_ad._current_level < 0


def _lora_present(lora_a, lora_b) -> bool:
    return lora_a is not None and lora_b is not None and lora_a.shape[0] > 0


def _lora_term(x, lora_a, lora_b, scaling):
    """(x @ A^T @ B^T * s) in x's dtype (lora_layer.py:67)."""
    return x @ lora_a.to(x.dtype).T @ lora_b.to(x.dtype).T * scaling


def _lora_backward(dy, x, A, B, s, need_a, need_b, need_g):
    """Gradients of (x A^T) B^T * s in x's dtype, cast to the parameters':
    dv = dY * s, dB = dv^T (x A^T), dA = (dv B)^T x; and dv B (None where the
    torch path runs), which dX's LoRA term starts from.  The HIP kernels run in
    eager first-order backward passes; tracing, create_graph (whose result is
    differentiated again), forward-mode AD and batched gradients
    (is_grads_batched: dy without storage), fp32 and ranks past 64 run on torch."""
    if _plain_eager() and not torch.is_grad_enabled() and dy.dtype == x.dtype and torch._C._has_storage(dy) and \
            ops.lora_grads_supported(x, A):
        return ops.lora_grads(x, dy, A, B, s, need_a, need_b, need_g)
    da = db = None
    dt = x.dtype
    x2 = x.reshape(-1, x.shape[-1])
    dv = dy.reshape(-1, dy.shape[-1]).to(dt) * s
    if need_b:
        u = x2 @ A.to(dt).T
        db = (dv.T @ u).to(B.dtype)
    if need_a:
        da = ((dv @ B.to(dt)).T @ x2).to(A.dtype)
    return da, db, None


class _FusedNF4LinearFunc(torch.autograd.Function):
    """y = x . W_deq^T + bias (+ LoRA) by the HIP kernels; backward gives dX
    (NF4 dX kernel, LoRA term fused) and the adapters' gradients.

    With LoRA dropout p > 0 the adapter reads drop(x) (lora_layer.py:67):
    the mask comes from torch's own dropout kernel (aten::native_dropout,
    the kernel nn.Dropout runs, so the random stream is the same), the
    forward passes drop(x) as the LoRA input of the fused kernels, and the
    dX kernel applies dropout's backward (mask / (1 - p)) to the adapter's
    input gradient in its epilogue."""

    @staticmethod
    def forward(ctx, x, lora_a, lora_b, bias, w: NF4Weight, scaling: float, dropout_p: float = 0.0):
        lora = _lora_present(lora_a, lora_b)
        xl = mask = None
        if lora and dropout_p > 0.0:
            xl, mask = torch.ops.aten.native_dropout(x, float(dropout_p), True)
        ctx.w = w
        ctx.scaling = float(scaling)
        ctx.lora = lora
        ctx.mask_scale = 1.0 / (1.0 - dropout_p) if mask is not None else 1.0
        ctx.save_for_backward(x if lora else None, lora_a if lora else None, lora_b if lora else None,
                              xl, mask)
        return torch_ops.call_nf4_linear(x, w.packed, w.scales, w.N, w.block_size, bias,
                                         lora_a=lora_a if lora else None, lora_b=lora_b if lora else None,
                                         scaling=scaling, lora_x=xl, **w.dq_kwargs())

    @staticmethod
    def backward(ctx, dy):
        x, A, B, xl, mask = ctx.saved_tensors
        w: NF4Weight = ctx.w
        s = ctx.scaling
        need_x, need_a, need_b = ctx.needs_input_grad[:3]
        dx = da = db = g = None
        grads = ctx.lora and (need_a or need_b)
        if grads:
            da, db, g = _lora_backward(dy, xl if xl is not None else x, A, B, s, need_a, need_b, need_x)
        if need_x:
            dx = torch_ops.call_nf4_linear_dx(dy, w.packed, w.scales, w.K, w.block_size,
                                              lora_a=A, lora_b=B, scaling=s, lora_mask=mask,
                                              mask_scale=ctx.mask_scale, lora_g=g, **w.dq_kwargs())
        return dx, da, db, None, None, None, None


class _FusedInt8LinearFunc(torch.autograd.Function):
    """y = x . (q * s)^T + bias by the HIP int8 kernels; backward dX =
    dY . RND(W_deq) (dequant_matmul.py:308-324) by the HIP int8 dX kernel."""

    @staticmethod
    def forward(ctx, x, bias, w: Int8Weight):
        ctx.w = w
        return torch_ops.call_int8_linear(x, w.q, w.scales, w.N, w.block_size, bias)

    @staticmethod
    def backward(ctx, dy):
        if not ctx.needs_input_grad[0]:
            return None, None, None
        w: Int8Weight = ctx.w
        return torch_ops.call_int8_linear_dx(dy, w.q, w.scales, w.K, w.block_size), None, None


def native_adapter(x, lora_a) -> bool:
    """Whether the adapter of an INT8 or FP8 layer runs on the LoRA kernels, both
    ways (eager, 16-bit activations, K a multiple of 64, rank <= 64, no autocast
    to another dtype, which torch's products would follow)."""
    return _plain_eager() and ops.lora_grads_supported(x, lora_a) and ops.lora_add_supported(x, lora_a) and \
        (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == x.dtype)


class _BaseLoRALinearFunc(torch.autograd.Function):
    """base(x) + (drop(x) A^T) B^T * s where base is a HIP linear without a LoRA
    epilogue (INT8, FP8): the term is added in place by the LoRA kernels, and
    the backward is the adapters' gradient kernels and base's dX with the
    adapter's input gradient in its epilogue.  base_dx(dy, A, B, s, g, mask,
    mask_scale) returns that dX, or None where it cannot include the term."""

    @staticmethod
    def forward(ctx, x, lora_a, lora_b, scaling: float, dropout_p: float, base, base_dx):
        xl, mask = x, None
        if dropout_p > 0.0:
            xl, mask = torch.ops.aten.native_dropout(x, float(dropout_p), True)
        ctx.base_dx = base_dx
        ctx.scaling = float(scaling)
        ctx.mask_scale = (1.0 / (1.0 - dropout_p) if dropout_p < 1.0 else 0.0) if mask is not None else 1.0
        ctx.save_for_backward(x, xl if mask is not None else None, lora_a, lora_b, mask)
        return ops.lora_add_(base(x), xl, lora_a, lora_b, scaling)

    @staticmethod
    def backward(ctx, dy):
        x, xl, A, B, mask = ctx.saved_tensors
        need_x, need_a, need_b = ctx.needs_input_grad[:3]
        if mask is None:
            xl = x
        elif torch.is_grad_enabled():  # create_graph: drop(x) as a function of x
            xl = x * (mask.to(x.dtype) * ctx.mask_scale)
        da, db, g = _lora_backward(dy, xl, A, B, ctx.scaling, need_a, need_b, need_x)
        dx = ctx.base_dx(dy, A, B, ctx.scaling, g, mask, ctx.mask_scale) if need_x else None
        return dx, da, db, None, None, None, None


def int8_lora_linear(x: torch.Tensor, w: Int8Weight, bias, lora_a, lora_b, scaling: float,
                     dropout_p: float = 0.0) -> torch.Tensor:
    """The INT8 linear plus the adapter's term, each rounded as the composed
    layers round them (lora_layer.py:58-70)."""
    if not native_adapter(x, lora_a):
        y = int8_linear(x, w, bias)
        xl = torch.nn.functional.dropout(x, dropout_p, True) if dropout_p > 0.0 else x
        return y + _lora_term(xl, lora_a, lora_b, scaling).to(y.dtype)
    nat.require_gpu(x, w.q)
    bias = bias.to(x.dtype) if bias is not None else None

    def base(x):
        return ops.int8_linear(x, w.q, w.scales, w.N, w.block_size, bias)

    def base_dx(dy, A, B, s, g, mask, mask_scale):
        if g is not None:
            return ops.int8_linear_dx(dy, w.q, w.scales, w.K, w.block_size, lora_a=A, lora_g=g, lora_mask=mask,
                                      mask_scale=mask_scale)
        return composed_dx(int8_dx(dy, w), dy, A, B, s, mask, mask_scale)

    return base_lora_linear(x, lora_a, lora_b, scaling, dropout_p, base, base_dx)


def base_lora_linear(x, lora_a, lora_b, scaling, dropout_p, base, base_dx):
    """_BaseLoRALinearFunc, or its forward alone where nothing is recorded."""
    if dropout_p == 0.0 and not (torch.is_grad_enabled() and
                                 (x.requires_grad or lora_a.requires_grad or lora_b.requires_grad)):
        return ops.lora_add_(base(x), x, lora_a, lora_b, scaling)
    return _BaseLoRALinearFunc.apply(x, lora_a, lora_b, float(scaling), float(dropout_p), base, base_dx)


def int8_dx(dy, w: Int8Weight):
    return torch_ops.call_int8_linear_dx(dy, w.q, w.scales, w.K, w.block_size)


def composed_dx(dx, dy, A, B, s, mask, mask_scale):
    """dx plus the adapter's input gradient ((dY s) B) A (times the dropout mask)
    by torch operators, which are differentiable again."""
    dt = dy.dtype
    t = (dy * s) @ B.to(dt) @ A.to(dt)
    return dx + (t * (mask.to(dt) * mask_scale) if mask is not None else t)


def _nothing_recorded(*inputs) -> bool:
    """Whether autograd records nothing for an op on these inputs, so that the
    forward can run without its autograd function: no gradient asked for, and
    neither tracing, a functorch transform nor forward-mode AD active (those go
    through the function, which accepts or refuses them)."""
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in inputs):
        return False
    return _plain_eager()


def nf4_linear(x: torch.Tensor, w: NF4Weight, bias: Optional[torch.Tensor] = None,
               lora_a: Optional[torch.Tensor] = None, lora_b: Optional[torch.Tensor] = None,
               scaling: float = 0.0, dropout_p: float = 0.0) -> torch.Tensor:
    """Autograd-aware NF4 linear (+ LoRA, its input through dropout of
    probability dropout_p when > 0) on the HIP kernels."""
    nat.require_gpu(x, w.packed)
    if not w.kernel_ok(x.dtype):
        raise TypeError(f"NF4 linear takes fp32/bf16/fp16 activations, got {x.dtype}")
    # the reference adds bias.to(x.dtype) (quant_linear.py:196)
    bias = bias.to(x.dtype) if bias is not None else None
    if dropout_p == 0.0 and _nothing_recorded(x, lora_a, lora_b, bias):
        return ops.nf4_linear(x, w.packed, w.scales, w.N, w.block_size, bias, lora_a=lora_a, lora_b=lora_b,
                              scaling=scaling, **w.dq_kwargs())
    return _FusedNF4LinearFunc.apply(x, lora_a, lora_b, bias, w, scaling, float(dropout_p))


def int8_linear(x: torch.Tensor, w: Int8Weight, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Autograd-aware INT8 linear on the HIP kernels."""
    nat.require_gpu(x, w.q)
    if not w.kernel_ok(x.dtype):
        raise TypeError(f"INT8 linear takes fp32/bf16/fp16 activations, got {x.dtype}")
    bias = bias.to(x.dtype) if bias is not None else None
    if _nothing_recorded(x, bias):
        return ops.int8_linear(x, w.q, w.scales, w.N, w.block_size, bias)
    return _FusedInt8LinearFunc.apply(x, bias, w)


def fused_dequant_nf4_matmul(x: torch.Tensor, w_packed: torch.Tensor, scales: torch.Tensor,
                             bias: Optional[torch.Tensor] = None, block_size: int = 64) -> torch.Tensor:
    """y = x . dequant_nf4(w)^T + bias (dequant_matmul.py:367-376).  w_packed
    is 1-D flat (N = numel * 2 // K) or 2-D [N, K // 2]; output has x's dtype
    and leading dims; differentiable in x (backward returns dX only)."""
    K = x.shape[-1]
    N = w_packed.numel() * 2 // K if w_packed.dim() == 1 else w_packed.shape[0]
    return nf4_linear(x, NF4Weight(w_packed.reshape(-1), scales, N, K, block_size), bias)


def fused_dequant_int8_matmul(x: torch.Tensor, w_int8: torch.Tensor, scales: torch.Tensor,
                              bias: Optional[torch.Tensor] = None, block_size: int = 64) -> torch.Tensor:
    """y = x . dequant_int8(w)^T + bias (dequant_matmul.py:356-365).  w_int8 is
    [N, K]; like dequantize_int8, one scale per row when scales.numel() == N,
    otherwise blockwise over the flat weight."""
    K = x.shape[-1]
    if w_int8.dim() != 2:
        raise ValueError(f"w_int8 must be [N, K], got shape {tuple(w_int8.shape)}")
    N = w_int8.shape[0]
    per_row = scales.numel() == N
    w = Int8Weight(w_int8, scales, N, K, 0 if per_row else block_size)
    return int8_linear(x, w, bias)
