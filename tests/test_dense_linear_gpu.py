"""Linears that decode the weight once into scratch memory and multiply by the
dense MFMA GEMM (csrc/dense_gemm.hip): tile edges, K splits, reduction lengths
that are padded, every decode kernel, the LoRA and dropout epilogues, against the
oracle at the tolerance of the other linears (16-bit results: rtol = atol = 1e-2,
fp32 1e-3, gradients relative to the largest).  FORWARD and the INT8 shapes run on
128 x 128 tiles; LARGE reaches the 256 x 256 ones, with operands whose sums are
exact in fp32, so that every bit is compared.

The entry points are called with scratch memory of the size the library
reports for the dense path, whatever the row count, through the C ABI."""
import ctypes

import pytest
import torch

from oracle import qlora_ref as R
from rocm_qlora import _native as nat
from rocm_qlora import ops
from rocm_qlora.quantization import dequantize_int4, double_quantize, quantize_int4, quantize_int8

pytestmark = pytest.mark.gpu
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g) * scale


def _check(got, ref, relative=False):
    tol = 1e-3 if got.dtype == torch.float32 else 1e-2
    got, ref = got.detach().cpu().float(), ref.detach().float()
    assert got.shape == ref.shape
    atol = tol * (float(ref.abs().max()) if relative else 1.0)
    err = (got - ref).abs()
    bad = err > atol + tol * ref.abs()
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tol; max err {float(err.max()):.4g}"


# (M, K, N, block, rank, dtype, storage): rows and columns around multiples of 128, one to many 64-k steps (prefetches past the end; odd step
# counts), splits (few tiles, long K), lengths padded to 64, blocks of 32 and
# blocks that straddle rows, ranks of one and two epilogue steps and past 64
FORWARD = [
    (17, 64, 64, 64, 0, "bf16", "f32"),
    (129, 128, 130, 64, 8, "bf16", "f32"),
    (256, 192, 256, 64, 16, "fp16", "f32"),
    (257, 320, 255, 64, 12, "bf16", "dq"),
    (300, 2048, 96, 128, 80, "bf16", "bf16"),
    (40, 320, 200, 32, 16, "bf16", "f32"),
    (33, 37, 73, 64, 4, "fp16", "f32"),
    (5, 1000, 301, 64, 12, "bf16", "dq"),
    (1, 130, 1, 64, 1, "bf16", "f32"),
    (1100, 4096, 512, 64, 64, "bf16", "f32"),
    (17, 64, 64, 64, 0, "fp32", "f32"),
    (130, 96, 129, 32, 8, "fp32", "f32"),
    (257, 320, 255, 64, 12, "fp32", "dq"),
    (5, 1000, 301, 64, 70, "fp32", "bf16"),
    (300, 2048, 512, 64, 33, "fp32", "f32"),
]


def _weight(g, N, K, block, storage, dev):
    w = _randn(g, N, K, scale=0.02)
    if storage == "dq":
        st = double_quantize(w.to(dev), block, 256)
        kw = dict(c2=st.c2, c2_scales=st.c2_scales, blocksize_2=256, use_fp8_c2=st.use_fp8_c2)
        wf = R.double_dequantize(st.W_quant.cpu(), st.c2.cpu(), st.c2_scales.cpu().reshape(-1), (N, K), block, 256,
                                 st.use_fp8_c2)
        return st.W_quant, None, kw, wf
    packed, s = quantize_int4(w.to(dev).to(torch.bfloat16 if storage == "bf16" else torch.float32), block)
    s = s.reshape(-1)
    return packed, s, {}, R.dequantize_int4(packed.cpu(), s.cpu(), block)[:N * K].reshape(N, K)


@pytest.fixture
def always_dense(monkeypatch):
    """The wrappers with the rule set aside: scratch memory for every call and
    the C entry point it belongs to (a block size no fused kernel takes is
    reported to the size query, so that it answers for the dense path)."""
    real = ops._scratch

    def scratch(fn, dev, *args):
        if "scratch" not in fn:
            return real(fn, dev, *args)
        nb = ctypes.c_int64(0)
        args = list(args)
        args[4] = 7
        nat.call(fn, *args, ctypes.byref(nb))
        assert nb.value > 0
        return torch.full((nb.value,), 0xFF, dtype=torch.uint8, device=dev)  # NaN patterns: contents must not matter

    monkeypatch.setattr(ops, "_scratch", scratch)


@pytest.mark.parametrize("M,K,N,block,rank,dtype,storage", FORWARD)
def test_dense_forward(dev, always_dense, M, K, N, block, rank, dtype, storage):
    print(f"dense forward {M} {K} {N} {block} {rank} {dtype} {storage}", flush=True)
    dt = DTYPES[dtype]
    g = torch.Generator().manual_seed(M + K + N)
    packed, s, kw, wf = _weight(g, N, K, block, storage, dev)
    x, bias = _randn(g, M, K).to(dt), _randn(g, N, scale=0.1)
    a, b = _randn(g, rank, K, scale=0.05), _randn(g, N, rank, scale=0.05)
    y = ops.nf4_linear(x.to(dev), packed, s, N, block, bias.to(dt).to(dev), lora_a=a.to(dev) if rank else None,
                       lora_b=b.to(dev) if rank else None, scaling=0.5, **kw)
    ref = R.quant_linear_forward(x, wf.reshape(-1), bias, N, K)
    if rank:
        ref = R.lora_forward(x, ref, a, b, 0.5)
    _check(y, ref)


@pytest.mark.parametrize("M,K,N,block,rank,dtype,storage,masked",
                         [(*c, m) for c in FORWARD for m in (False, True) if c[4] or not m])
def test_dense_dx(dev, always_dense, M, K, N, block, rank, dtype, storage, masked):
    print(f"dense dx {M} {K} {N} {block} {rank} {dtype} {storage} {masked}", flush=True)
    dt = DTYPES[dtype]
    g = torch.Generator().manual_seed(M + K + N + 1)
    packed, s, kw, wf = _weight(g, N, K, block, storage, dev)
    dy = _randn(g, M, N, scale=0.05).to(dt)
    a, b = _randn(g, rank, K, scale=0.05), _randn(g, N, rank, scale=0.05)
    mask = torch.rand(M, K, generator=g) < 0.8
    dx = ops.nf4_linear_dx(dy.to(dev), packed, s, K, block, lora_a=a.to(dev) if rank else None,
                           lora_b=b.to(dev) if rank else None, scaling=0.5,
                           lora_mask=mask.to(dev) if masked else None, mask_scale=1.25 if masked else 1.0, **kw)
    ref = dy.float() @ wf.to(dt).float()
    ref = ref.to(dt)
    if rank:
        l = (dy * 0.5) @ b.to(dt) @ a.to(dt)
        ref = ref + (l * (mask.to(dt) * 1.25) if masked else l)
    _check(dx, ref, relative=True)


@pytest.mark.parametrize("M,K,N,block", [(17, 64, 64, 0), (130, 320, 192, 64), (300, 129, 257, 0), (20, 96, 64, 32),
                                         (257, 2048, 96, 128), (3, 73, 37, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_dense_int8(dev, always_dense, M, K, N, block, dtype):
    print(f"dense int8 {M} {K} {N} {block} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + K + N + 2)
    w = _randn(g, N, K, scale=0.02).to(dev)
    q, s = quantize_int8(w, per_channel=True) if block == 0 else quantize_int8(w, block)
    wf = R.dequantize_int8(q.cpu(), s.cpu().reshape(-1), block or 64).reshape(-1)[:N * K].reshape(N, K).to(dtype)
    x, dy, bias = _randn(g, M, K).to(dtype), _randn(g, M, N, scale=0.05).to(dtype), _randn(g, N, scale=0.1)
    y = ops.int8_linear(x.to(dev), q, s, N, block, bias.to(dtype).to(dev))
    _check(y, torch.nn.functional.linear(x, wf, bias.to(dtype)))
    dx = ops.int8_linear_dx(dy.to(dev), q, s, K, block)
    _check(dx, (dy.float() @ wf.float()).to(dtype), relative=True)


def test_dense_rule_matches_general_path(dev):
    """Calls that the rule sends to the dense path against the same calls
    without scratch memory (the fused and generic kernels), strided and
    misaligned activations among them: the operands round alike, so the
    results differ by the order of fp32 sums and its effect on one rounding."""
    g = torch.Generator().manual_seed(5)
    N, K, M = 4096, 1024, 4096
    w = _randn(g, N, K, scale=0.02).to(dev)
    packed, s = quantize_int4(w, 64)
    q, qs = quantize_int8(w, 64)
    wide = _randn(g, M, K + 4).to(torch.bfloat16).to(dev)
    dy = _randn(g, M, N, scale=0.05).to(torch.bfloat16).to(dev)
    real = ops._scratch
    for x in (wide[:, :K].contiguous(), wide[:, :K], wide[:, 1:K + 1]):
        calls = [lambda: ops.nf4_linear(x, packed, s, N, 64), lambda: ops.nf4_linear_dx(dy, packed, s, K, 64),
                 lambda: ops.int8_linear(x, q, qs, N, 64), lambda: ops.int8_linear_dx(dy, q, qs, K, 64)]
        for i, call in enumerate(calls):
            sizes = []

            def spy(fn, dev_, *args):
                r = real(fn, dev_, *args)
                if "scratch" in fn:
                    sizes.append(0 if r is None else r.numel())
                return r

            ops._scratch = spy
            try:
                got = call()
                assert sizes and sizes[0] > 0, f"call {i} is expected on the dense path"
                ops._scratch = lambda fn, dev_, *args: None if "scratch" in fn else real(fn, dev_, *args)
                ref = call()
            finally:
                ops._scratch = real
            # one bf16 rounding may fall the other way: 2^-8 of the value
            d = (got.float() - ref.float()).abs()
            assert bool((d <= 2.0 ** -7 * ref.float().abs() + 1e-5 * float(ref.abs().max())).all()), f"call {i}"


# (M, R, C, rank, dtype, bias) and what the plan makes of them: tile edge, whole
# tiles, split tiles, splits.  256 x 256 tiles with ragged rows and columns; 11
# (the fewest the plan gives them) and 12 steps; a padded reduction; one split
# count each of whole tiles mixed with split ones; split tiles alone, with an odd
# number of steps a split.  And the 128 x 128 tiles' mix.
LARGE = [
    (4000, 700, 4001, 0, "bf16", True, (256, 256, 0, 1)),
    (3841, 768, 3841, 12, "fp16", True, (256, 256, 0, 1)),
    (4097, 3100, 4097, 16, "bf16", False, (256, 256, 33, 4)),
    (5000, 2560, 3600, 64, "bf16", True, (256, 256, 44, 4)),
    (4097, 4096, 4609, 16, "fp16", False, (256, 256, 67, 2)),
    (700, 11001, 4000, 8, "bf16", False, (256, 0, 48, 4)),
    (1290, 4096, 4096, 16, "bf16", True, (128, 256, 96, 2)),
]


def _tile_plan(dtype, M, C, R):
    out = (ctypes.c_int32 * 4)()
    nat.call("rq_dense_tile_plan", nat.dtype_code(DTYPES[dtype]), M, C, R, out)
    return tuple(out)


def _ints(g, dev, lo, hi, *shape):
    return torch.randint(lo, hi + 1, shape, generator=g, device=dev).double()


def _whole_weight(g, dev, N, K):
    """An NF4 weight of the values -2, -1, 0, 1, 2: codes of -1, 0 and 1 and absmax 1
    or 2."""
    code = torch.tensor([0, 7, 15], dtype=torch.uint8, device=dev)[torch.randint(0, 3, (N * K + N * K % 2,), generator=g, device=dev)]
    absmax = torch.randint(1, 3, (-(-N * K // 64),), generator=g, device=dev).float()
    value = torch.tensor([-1.0, 0.0, 1.0], dtype=torch.float64, device=dev)[(code.long() + 7) // 8]
    w = (value[:N * K] * absmax.double().repeat_interleave(64)[:N * K]).reshape(N, K)
    return code[0::2] | (code[1::2] << 4), absmax, w


@pytest.mark.parametrize("M,R,C,rank,dtype,bias,plan", LARGE)
def test_dense_tiles_forward_exact(dev, always_dense, M, R, C, rank, dtype, bias, plan):
    print(f"dense exact forward {M} {R} {C} {rank} {dtype} {plan}", flush=True)
    assert _tile_plan(dtype, M, C, R) == plan
    dt, g = DTYPES[dtype], torch.Generator(device=dev).manual_seed(M + R + C)

    def rnd(t):
        return t.to(dt).double()

    packed, absmax, w = _whole_weight(g, dev, C, R)
    x, b = _ints(g, dev, -3, 3, M, R), _ints(g, dev, -500, 500, C)
    la, lb = _ints(g, dev, -2, 2, rank, R), _ints(g, dev, -1, 1, C, rank)
    y = ops.nf4_linear(x.to(dt), packed, absmax, C, 64, b.to(dt) if bias else None, lora_a=la.float() if rank else None,
                       lora_b=lb.float() if rank else None, scaling=0.5)
    ref = rnd(x @ w.T + (rnd(b) if bias else 0.0))
    if rank:
        ref = rnd(ref + rnd(rnd(rnd(x @ la.T) @ lb.T) * 0.5))
    assert float((x @ w.T).abs().max()) > 256  # past bf16's 8 bits
    assert torch.equal(y.double(), ref)


@pytest.mark.parametrize("M,R,C,rank,dtype,masked,plan", [(*c[:5], m, c[6]) for c in LARGE for m in (False, True) if c[3] or not m])
def test_dense_tiles_dx_exact(dev, always_dense, M, R, C, rank, dtype, masked, plan):
    print(f"dense exact dx {M} {R} {C} {rank} {dtype} {masked} {plan}", flush=True)
    assert _tile_plan(dtype, M, C, R) == plan
    dt, g = DTYPES[dtype], torch.Generator(device=dev).manual_seed(M + R + C + 1)

    def rnd(t):
        return t.to(dt).double()

    packed, absmax, w = _whole_weight(g, dev, R, C)  # [N, K] = [R, C]
    dy = _ints(g, dev, -3, 3, M, R)
    la, lb = _ints(g, dev, -1, 1, rank, C), _ints(g, dev, -2, 2, R, rank)
    mask = torch.rand(M, C, generator=g, device=dev) < 0.8
    dx = ops.nf4_linear_dx(dy.to(dt), packed, absmax, C, 64, lora_a=la.float() if rank else None,
                           lora_b=lb.float() if rank else None, scaling=0.5, lora_mask=mask if masked else None,
                           mask_scale=1.25 if masked else 1.0)
    ref = rnd(dy @ w)
    if rank:
        term = rnd(rnd(rnd(dy * 0.5) @ lb) @ la)
        ref = rnd(ref + (rnd(term * mask * 1.25) if masked else term))
    assert torch.equal(dx.double(), ref)


@pytest.mark.parametrize("M,K,N", [(1000, 1024, 4096), (256, 4096, 4096), (1000, 4096, 4096), (96, 4096, 14336),
                                   (1000, 14336, 1024), (300, 512, 512), (200, 1000, 1501), (700, 96, 2048)])
def test_dense_fp32_is_no_less_precise(dev, monkeypatch, M, K, N):
    """fp32 forward and dX: the dense product's error against float64 is not above
    that of the kernels over the stored codes (2-norms over 10^5 values and more,
    which vary by less than 2 % from draw to draw)."""
    print(f"dense fp32 precision {M} {K} {N}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + K + N)
    packed, s = quantize_int4(torch.randn(N, K, generator=g, device=dev) * 0.02, 64)
    w = dequantize_int4(packed, s, 64).reshape(-1)[:N * K].reshape(N, K).double()
    x, dy = torch.randn(M, K, generator=g, device=dev), torch.randn(M, N, generator=g, device=dev)
    real = ops._scratch

    def dense(fn, d, *args):
        if "scratch" not in fn:
            return real(fn, d, *args)
        return torch.empty(ops._bytes(fn, d.index, *args[:4], 7, *args[5:]), dtype=torch.uint8, device=d)

    def errors(route):
        monkeypatch.setattr(ops, "_scratch", route)
        return [float((got.double() - ref).norm() / ref.norm()) for got, ref in
                ((ops.nf4_linear(x, packed, s, N, 64), x.double() @ w.T), (ops.nf4_linear_dx(dy, packed, s, K, 64), dy.double() @ w))]

    codes = errors(lambda fn, d, *args: None if "scratch" in fn else real(fn, d, *args))
    for name, a, b in zip(("y", "dx"), errors(dense), codes):
        assert a <= 1.02 * b, f"{name}: {a:.3g} dense, {b:.3g} from the codes"


def test_replayed_training_operands(dev):
    """One graph with the calls of training steps (dense products with and without
    split tiles, the adapters' gradients, INT8 dX with the adapter's term, the
    adapter added in place), replayed among eager calls and changed inputs: the
    eager bits each time."""
    g = torch.Generator(device=dev).manual_seed(8)

    def randn(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device=dev) * scale

    M, K, N, r = 1290, 4096, 4096, 16
    packed, s = quantize_int4(randn(N, K, scale=0.02), 64)
    q, qs = quantize_int8(randn(N, K, scale=0.02), 64)
    x, dy = randn(M, K).bfloat16(), randn(M, N, scale=0.05).bfloat16()
    a, b = randn(r, K, scale=0.02), randn(N, r, scale=0.05)

    def calls():
        da, db, gg = ops.lora_grads(x, dy, a, b, 2.0, True, True, True)
        y8 = ops.lora_add_(ops.int8_linear(x, q, qs, N, 64), x, a, b, 2.0)
        xf = x[:48].float()
        return (ops.nf4_linear(x[:300], packed, s, N, 64, lora_a=a, lora_b=b, scaling=2.0),
                ops.nf4_linear_dx(dy, packed, s, K, 64, lora_a=a, lora_b=b, scaling=2.0, lora_g=gg),
                ops.int8_linear_dx(dy, q, qs, K, 64, lora_a=a, lora_g=gg), da, db, y8,
                ops.nf4_linear(xf.repeat(4, 1), packed, s, N, 64, lora_a=a, lora_b=b, scaling=2.0),
                ops.nf4_linear(x, packed, s, N, 64, lora_a=a, lora_b=b, scaling=2.0))

    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        calls()
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            out = calls()
    torch.cuda.synchronize()
    for _ in range(4):
        x.copy_(randn(M, K))
        dy.copy_(randn(M, N, scale=0.05))
        eager = calls()
        [o.fill_(float("nan")) for o in out]
        graph.replay()
        again = calls()
        torch.cuda.synchronize()
        for i, (o, e, f) in enumerate(zip(out, eager, again)):
            assert torch.equal(o, e) and torch.equal(e, f), i
