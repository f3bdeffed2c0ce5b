"""The adapters' gradient kernels (csrc/lora_grad.hip): rows around the 32-row
steps and the row splits, columns around the 128-wide tiles and the padded
lengths, every rank block count, against the reference's torch expressions in
float64 on the same 16-bit inputs.

Bound: every intermediate (dv, u, g) and the result is rounded once to the
activation dtype, as the reference's are; an fp32 sum in another order moves a
rounding by at most one unit.  So each result lies within 3 roundings of the
float64 value in the 2-norm: 3 * 2^-9 (bf16) or 3 * 2^-12 (fp16; small values
also lose to its subnormals)."""
import pytest
import torch

from rocm_qlora import ops

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.mark.parametrize("M,K,N,rank,dtype", [
    (1, 64, 64, 8, "bf16"), (31, 128, 192, 16, "fp16"), (33, 100, 130, 12, "bf16"), (128, 320, 64, 17, "bf16"),
    (129, 64, 1000, 33, "bf16"), (300, 37, 73, 64, "fp16"), (2048, 512, 256, 64, "bf16"), (1500, 4096, 128, 48, "fp16"),
])
@pytest.mark.parametrize("lora32", [True, False])
def test_lora_grads(dev, M, K, N, rank, dtype, lora32):
    print(f"lora grads {M} {K} {N} {rank} {dtype} {lora32}", flush=True)
    dt = DT[dtype]
    g = torch.Generator().manual_seed(M + K + N + rank)
    x, dy = torch.randn(M, K, generator=g).to(dt), torch.randn(M, N, generator=g).to(dt)
    a, b = torch.randn(rank, K, generator=g) / K ** 0.5, torch.randn(N, rank, generator=g) / N ** 0.5
    if not lora32:
        a, b = a.to(dt), b.to(dt)
    s = 0.75
    da, db, gg = ops.lora_grads(x.to(dev), dy.to(dev), a.to(dev), b.to(dev), s, True, True, True)
    assert da.dtype == a.dtype and db.dtype == b.dtype and da.shape == a.shape and db.shape == b.shape
    xd, dyd, ad, bd = x.double(), dy.double(), a.to(dt).double(), b.to(dt).double()
    u, gv = (xd @ ad.T), s * dyd @ bd
    tol = 3 * 2.0 ** (-9 if dtype == "bf16" else -12)
    for name, got, ref in (("dA", da, gv.T @ xd), ("dB", db, s * dyd.T @ u), ("g", gg[:, :rank], gv)):
        err = float((got.cpu().double() - ref).norm() / ref.norm())
        assert err <= tol, f"{name}: {err:.2e} > {tol:.2e}"
    assert not gg[:, rank:].any()


@pytest.mark.parametrize("M,K,N,rank,dtype", [(4096, 4096, 14336, 64, "bf16"), (2048, 1024, 4096, 64, "fp16"),
                                              (333, 1000, 1501, 12, "bf16"), (1024, 4096, 4096, 16, "bf16")])
def test_lora_grads_exact_sums(dev, M, K, N, rank, dtype):
    """Small whole numbers, whose sums are exact in fp32 in any order: every bit
    equals the torch expressions of the adapter's gradients in float64 with one
    rounding to the activation dtype after each of them, so rounding points and
    widths are theirs and other inputs can differ by the order of the sums alone.
    (|u|, |g| stay near 2^8 to 2^10, past bf16's 8 bits, and the last sums below
    2^24.)"""
    print(f"lora grads, exact sums {M} {K} {N} {rank} {dtype}", flush=True)
    dt = DT[dtype]
    g = torch.Generator(device=dev).manual_seed(M + rank)

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, generator=g, device=dev).float()

    big = 4 if dtype == "bf16" else 2  # fp16: the sums stay below its largest value
    x, dy = ints(-1, 1, M, K).to(dt), ints(-1, 1, M, N).to(dt)
    a, b, s = ints(-big, big, rank, K), ints(-big, big, N, rank), 0.5
    da, db, gg = ops.lora_grads(x, dy, a, b, s, True, True, True)
    dv = (dy.double() * s).to(dt).double()
    u, gv = (x.double() @ a.double().T).to(dt).double(), (dv @ b.double()).to(dt).double()
    sa, sb = gv.T @ x.double(), dv.T @ u
    assert max(float(t.abs().max()) for t in (sa, sb)) < 2.0 ** 24 and float(u.abs().max()) > 2 ** 7
    assert torch.equal(gg[:, :rank].double(), gv) and not gg[:, rank:].any()
    assert torch.equal(da, sa.to(dt).float()) and torch.equal(db, sb.to(dt).float())


def test_lora_grads_strided_and_partial(dev):
    """Strided rows (16-byte aligned and not) give the same bits as packed
    ones, and each gradient alone the same as all together."""
    g = torch.Generator().manual_seed(3)
    M, K, N, r = 200, 128, 192, 16
    xw, yw = torch.randn(M, K + 9, generator=g).bfloat16().to(dev), torch.randn(M, N + 9, generator=g).bfloat16().to(dev)
    a, b = torch.randn(r, K, generator=g).to(dev), torch.randn(N, r + 3, generator=g).to(dev)[:, :r]
    for o in (0, 1, 8):
        x, y = xw[:, o:o + K], yw[:, o:o + N]
        ref = ops.lora_grads(x.contiguous(), y.contiguous(), a, b.contiguous(), 2.0, True, True, True)
        got = ops.lora_grads(x, y, a, b, 2.0, True, True, True)
        alone = (ops.lora_grads(x, y, a, b, 2.0, True, False)[0], ops.lora_grads(x, y, a, b, 2.0, False, True)[1])
        assert all(torch.equal(p, q) for p, q in zip(ref, got))
        assert torch.equal(alone[0], ref[0]) and torch.equal(alone[1], ref[1])


@pytest.mark.parametrize("M,K,N,rank,dtype", [(1, 64, 8, 8, "bf16"), (31, 128, 255, 17, "fp16"), (33, 320, 256, 16, "bf16"),
                                              (100, 4096, 300, 80, "bf16"), (300, 192, 1000, 64, "fp16")])
@pytest.mark.parametrize("lora32", [True, False])
def test_lora_add(dev, M, K, N, rank, dtype, lora32):
    """y += term in place: 32-row and 256-column tile edges, rows that are not
    16-byte aligned (N odd), ranks of one to several MFMA steps.  Each of the
    four roundings (u, the product, the scaling, the sum) is the reference's;
    bound 4 * 2^-9 (2^-12) of the result."""
    print(f"lora add {M} {K} {N} {rank} {dtype} {lora32}", flush=True)
    dt = DT[dtype]
    g = torch.Generator().manual_seed(M + K + N + rank)
    x, y = torch.randn(M, K, generator=g).to(dt), torch.randn(M, N, generator=g).to(dt)
    a, b = torch.randn(rank, K, generator=g) / K ** 0.5, torch.randn(N, rank, generator=g) / rank ** 0.5
    if not lora32:
        a, b = a.to(dt), b.to(dt)
    got = y.to(dev).clone()
    out = ops.lora_add_(got, x.to(dev), a.to(dev), b.to(dev), 0.75)
    assert out is got
    ref = y.double() + 0.75 * (x.double() @ a.to(dt).double().T) @ b.to(dt).double().T
    err = float((got.cpu().double() - ref).norm() / ref.norm())
    assert err <= 4 * 2.0 ** (-9 if dtype == "bf16" else -12), err


@pytest.mark.parametrize("kind", ["int8", "fp8_nf4", "fp8_int8"])
@pytest.mark.parametrize("p", [0.0, 0.25])
@pytest.mark.parametrize("M", [5, 40])
def test_byte_layers_with_adapter(dev, kind, p, M):
    """LoRALinear on an INT8 layer and FP8LinearWrapper: output and gradients of
    the fused adapter path against the same module composed by torch (its own
    path under create_graph), with and without dropout (same seed, same mask).
    The composed path rounds alike; sums in another order move a rounding by
    one unit: 2^-7 of the value plus 2^-7 of the rms covers two such."""
    import torch.nn as nn
    from rocm_qlora import LoRALinear, QuantLinear
    from rocm_qlora.fp8 import FP8LinearWrapper
    from rocm_qlora.kernels import dequant_matmul as dm
    torch.manual_seed(7)
    layer = LoRALinear(QuantLinear.from_linear(nn.Linear(192, 136).to(dev), bits=4 if kind == "fp8_nf4" else 8, block_size=64),
                       r=12, lora_alpha=24, lora_dropout=p).to(dev)
    with torch.no_grad():
        layer.lora_B.normal_(0, 0.05)
    module = layer if kind == "int8" else FP8LinearWrapper(layer)
    x = torch.randn(M, 192, device=dev, dtype=torch.bfloat16)
    dy = torch.randn(M, 136, device=dev, dtype=torch.bfloat16)

    def run():
        torch.manual_seed(11)
        xi = x.clone().requires_grad_(True)
        y = module(xi)
        return [y.detach(), *torch.autograd.grad(y, (xi, layer.lora_A, layer.lora_B), dy)]

    got = run()
    real = dm.native_adapter
    dm.native_adapter = lambda *a: False
    try:
        ref = run()
    finally:
        dm.native_adapter = real
    for name, a, b in zip(("y", "dx", "dA", "dB"), got, ref):
        assert a.dtype == b.dtype and a.shape == b.shape
        d, f = (a.float() - b.float()).abs(), b.float()
        assert bool((d <= 2.0 ** -7 * (f.abs() + f.square().mean().sqrt())).all()), (name, float(d.max()))


def _int8_layer(dev, K, N, r, dropout):
    from rocm_qlora import LoRALinear, QuantLinear
    g = torch.Generator().manual_seed(9)
    lin = torch.nn.Linear(K, N, bias=False)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(N, K, generator=g) * 0.02)
    layer = LoRALinear(QuantLinear.from_linear(lin.to(dev), bits=8), r=r, lora_alpha=2 * r, lora_dropout=dropout).to(dev)
    with torch.no_grad():
        layer.lora_B.copy_(torch.randn(N, r, generator=g) * 0.1)
    return layer.train()


@pytest.mark.parametrize("p", [0.0, 0.5, 1.0])
def test_int8_second_derivative_through_dropout(dev, p):
    """dA = s (dY B)^T drop(x) differentiated again: d<dA, V>/dx = s (dY B) V times
    the dropout mask.  Bound: four bf16 roundings."""
    K, N, r, M = 128, 192, 8, 40
    layer = _int8_layer(dev, K, N, r, p)
    g = torch.Generator().manual_seed(1)
    x = torch.randn(M, K, generator=g).bfloat16().to(dev).requires_grad_()
    dy = torch.randn(M, N, generator=g).bfloat16().to(dev)
    v = torch.randn(r, K, generator=g).to(dev)
    torch.manual_seed(5)
    y = layer(x)
    torch.manual_seed(5)
    keep = torch.nn.functional.dropout(torch.ones_like(x), p, True) if p else torch.ones_like(x)
    (da,) = torch.autograd.grad(y, layer.lora_A, dy, create_graph=True)
    (gx,) = torch.autograd.grad((da * v).sum(), x)
    ref = (layer.scaling * (dy.float() @ layer.lora_B.float()) @ v) * keep.float()
    assert (gx.float() - ref).norm() <= 4 * 2.0 ** -9 * ref.norm()


def test_linears_without_room_for_the_decoded_weight(dev, monkeypatch):
    """A GPU too full for the decoded weight: the other route's results, which
    differ from the dense route's by the order of fp32 sums (one bf16 rounding of
    each value, and one of the adapter's intermediates)."""
    layer = _int8_layer(dev, 256, 320, 16, 0.0)
    from rocm_qlora.quantization import quantize_int4
    g = torch.Generator().manual_seed(2)
    w = (torch.randn(1000, 333, generator=g) * 0.02).to(dev)
    packed, absmax = quantize_int4(w, 64)
    x, x4 = torch.randn(70, 256, generator=g).bfloat16().to(dev).requires_grad_(), torch.randn(70, 333, generator=g).bfloat16().to(dev)
    dy, dy4 = torch.randn(70, 320, generator=g).bfloat16().to(dev), torch.randn(70, 1000, generator=g).bfloat16().to(dev)

    def call():
        y = layer(x)
        return (y.detach(), torch.autograd.grad(y, x, dy)[0], ops.nf4_linear(x4, packed, absmax, 1000, 64),
                ops.nf4_linear_dx(dy4, packed, absmax, 333, 64))

    ref = call()
    real = ops._scratch

    def full(size_fn, d, *args):
        if size_fn.endswith("linear_scratch_size") or size_fn.endswith("linear_dx_scratch_size"):
            raise torch.OutOfMemoryError("full")
        return real(size_fn, d, *args)

    monkeypatch.setattr(ops, "_scratch", full)
    for a, b in zip(call(), ref):
        assert (a.float() - b.float()).norm() <= 3 * 2.0 ** -9 * b.float().norm()
