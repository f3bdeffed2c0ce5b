"""Which route the library's size queries give a call (scratch bytes: decode the
weight once and multiply densely; 0: the kernel over the stored codes), at sizes
where both routes were timed and lie well apart.  The queries answer for 256
compute units where there is no GPU."""
import ctypes

import pytest

from rocm_qlora import _native as nat

BF16, F32 = nat.DTYPE_BF16, nat.DTYPE_F32


def _size(name, *args):
    n = ctypes.c_int64(-1)
    nat.call(name, *args, ctypes.byref(n))
    return n.value


# (M, K, N, dense), times fused / dense in us
FORWARD = [
    (128, 4096, 4096, False),    # 27.6 / 30.4
    (256, 4096, 4096, False),    # 27.6 / 37.3
    (512, 4096, 4096, False),    # 33.2 / 40.0
    (1536, 4096, 4096, False),   # 62.5 / 72.1
    (3072, 4096, 4096, True),    # 120 / 96.4
    (192, 14336, 4096, False),   # 58.9 / 78.9
    (1024, 14336, 4096, False),  # 130 / 139
    (2048, 14336, 4096, True),   # 242 / 213
    (768, 11008, 4096, False),   # 86.3 / 99.7
    (512, 4096, 14336, False),   # 68.6 / 88.0
    (1024, 4096, 14336, True),   # 135 / 120
    (512, 2048, 2048, False),    # 21.1 / 24.8
    (1024, 1024, 8192, False),   # 24.4 / 37.7
    (4096, 4096, 14336, True),   # 500 / 397
]
# dX from N to K columns
DX = [
    (256, 4096, 4096, True),     # 69.7 / 39.3
    (256, 11008, 4096, True),    # 71.5 / 56.0
    (4096, 4096, 14336, True),   # 520 / 368
]
INT8 = [
    (512, 1024, 8192, False),    # 20.2 / 28.1
    (1536, 4096, 4096, False),   # 62.8 / 72.8
    (2048, 3072, 3072, False),   # 48.8 / 61.1
    (256, 4096, 4096, True),     # 56.8 / 38.4
]
# (M, K, N, rank, dense), times row blocks / dense
FORWARD_F32 = [
    (64, 4096, 4096, 0, False),    # 49 / 64
    (96, 4096, 4096, 0, True),     # 74 / 64
    (48, 14336, 4096, 16, False),  # 137 / 190
    (64, 14336, 4096, 0, False),   # 149 / 177
    (128, 14336, 4096, 0, True),   # 298 / 178
    (64, 4096, 14336, 16, True),   # 241 / 198
    (128, 1024, 1024, 0, True),    # 51 / 25
    (256, 512, 512, 64, True),     # 256 / 36
]


@pytest.mark.parametrize("M,K,N,dense", FORWARD)
def test_nf4_forward_route(M, K, N, dense):
    for rank in (0, 16):
        assert (_size("rq_nf4_linear_scratch_size", BF16, M, K, N, 64, rank) > 0) == dense


@pytest.mark.parametrize("M,K,N,dense", DX)
def test_nf4_dx_route(M, K, N, dense):
    assert (_size("rq_nf4_linear_dx_scratch_size", BF16, M, N, K, 64, 0) > 0) == dense


@pytest.mark.parametrize("M,K,N,dense", INT8)
def test_int8_forward_route(M, K, N, dense):
    assert (_size("rq_int8_linear_scratch_size", BF16, M, K, N, 64, 0, 0) > 0) == dense


@pytest.mark.parametrize("M,K,N,rank,dense", FORWARD_F32)
def test_nf4_forward_fp32_route(M, K, N, rank, dense):
    assert (_size("rq_nf4_linear_scratch_size", F32, M, K, N, 64, rank) > 0) == dense


@pytest.mark.parametrize("M,K,N,rank", [(17, 4096, 1024, 0), (48, 4096, 14336, 16), (48, 4096, 128256, 16), (64, 4096, 128256, 0),
                                        (64, 4096, 128256, 64), (64, 16384, 16384, 64), (33, 1024, 512, 0)])
def test_skinny_memory(M, K, N, rank):
    """The skinny kernel's splits, past 1.5 MiB, live in scratch memory of at most 128
    MiB, freed after the call; the workspace, which callers keep, holds what the fused GEMM
    needs (its K splits' tiles, at most one per compute unit) and the area the
    splits are counted in."""
    ws, scratch = _size("rq_nf4_linear_workspace_size", BF16, M, K, N, rank), _size("rq_nf4_linear_scratch_size", BF16, M, K, N, 64, rank)
    assert (131328 if (M, N) != (64, 128256) else 0) <= ws <= 131328 + 256 * 256 * 128 * 4 + (2 << 20)
    assert scratch <= 128 << 20
    # splits x rows x columns of fp32, or none: too much, or little enough for the workspace
    assert scratch == 0 or scratch >= 4 * M * N
    assert (scratch == 0) == ((M, K, N) in ((64, 4096, 128256), (64, 16384, 16384), (17, 4096, 1024), (33, 1024, 512)))
