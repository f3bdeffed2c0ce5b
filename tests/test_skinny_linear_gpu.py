"""The skinny NF4 linear (csrc/skinny_linear.hip, 17 to 64 rows): row blocks of
16, the last segment partly past K, one to many K splits, both segment counts
per split, partial column groups, LoRA ranks up to 64, against the oracle at the
tolerance of the other 16-bit linears (rtol = atol = 1e-2); and the same bits
from three calls, whichever split counts itself last, and from replays of a graph."""
import pytest
import torch

from oracle import qlora_ref as R
from rocm_qlora import ops
from rocm_qlora.quantization import double_quantize, quantize_int4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,block,rank,dtype,dq", [
    (17, 64, 16, 64, 0, "bf16", False), (32, 320, 130, 64, 12, "bf16", False), (33, 256, 257, 256, 16, "fp16", False),
    (48, 1088, 300, 64, 64, "bf16", True), (49, 4096, 272, 128, 16, "bf16", False), (64, 2048, 512, 64, 33, "fp16", True),
    (40, 4096, 8192, 64, 8, "bf16", False), (64, 14336, 96, 64, 16, "bf16", False),
])
def test_skinny_linear(dev, M, K, N, block, rank, dtype, dq):
    print(f"skinny {M} {K} {N} {block} {rank} {dtype} {dq}", flush=True)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    g = torch.Generator().manual_seed(M + K + N)
    w = torch.randn(N, K, generator=g) * 0.02
    kw = {}
    if dq:
        st = double_quantize(w.to(dev), block, 256)
        packed, s = st.W_quant, None
        kw = dict(c2=st.c2, c2_scales=st.c2_scales, blocksize_2=256, use_fp8_c2=st.use_fp8_c2)
        wf = R.double_dequantize(st.W_quant.cpu(), st.c2.cpu(), st.c2_scales.cpu().reshape(-1), (N, K), block, 256,
                                 st.use_fp8_c2)
    else:
        packed, s = quantize_int4(w.to(dev), block)
        wf = R.dequantize_int4(packed.cpu(), s.cpu(), block)
    x, bias = torch.randn(M, K, generator=g).to(dt), torch.randn(N, generator=g) * 0.1
    a, b = torch.randn(rank, K, generator=g) * 0.02, torch.randn(N, rank, generator=g) * 0.05
    args = (x.to(dev), packed, s, N, block, bias.to(dt).to(dev))
    if rank:
        kw.update(lora_a=a.to(dev), lora_b=b.to(dev), scaling=0.5)
    outs = [ops.nf4_linear(*args, **kw) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    ref = R.quant_linear_forward(x, wf.reshape(-1), bias, N, K)
    if rank:
        ref = R.lora_forward(x, ref, a, b, 0.5)
    err = (outs[0].cpu().float() - ref.float()).abs()
    bad = err > 1e-2 + 1e-2 * ref.float().abs()
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tol; max err {float(err.max()):.4g}"


def test_skinny_linear_replayed(dev):
    """Two captured calls that share the capture's scratch memory and counters,
    replayed among eager calls on the same operands: the eager bits every time."""
    g = torch.Generator().manual_seed(4)
    calls = []
    for M, K, N in ((40, 4096, 512), (64, 2048, 1088)):
        packed, s = quantize_int4((torch.randn(N, K, generator=g) * 0.02).to(dev), 64)
        x = torch.randn(M, K, generator=g).bfloat16().to(dev)
        a, b = (torch.randn(16, K, generator=g) * 0.02).to(dev), (torch.randn(N, 16, generator=g) * 0.05).to(dev)
        calls.append(lambda x=x, packed=packed, s=s, N=N, a=a, b=b: ops.nf4_linear(x, packed, s, N, 64, lora_a=a, lora_b=b, scaling=0.5))
    ref = [c() for c in calls]
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        [c() for c in calls]
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            out = [c() for c in calls]
    torch.cuda.synchronize()
    for _ in range(4):
        [o.fill_(float("nan")) for o in out]
        graph.replay()
        eager = [c() for c in calls]
        torch.cuda.synchronize()
        assert all(torch.equal(o, r) and torch.equal(e, r) for o, e, r in zip(out, eager, ref))
