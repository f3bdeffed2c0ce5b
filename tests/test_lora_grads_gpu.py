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
