"""What a prompt leaves in pages of e4m3 is bytes, so the kernels of its step keep
the order of their sums: the same bits come out whichever of them a size has."""

import zlib

import numpy as np
import pytest
import torch

from llmapigateway_amd import ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _rows(rs, *shape, by=1.0):
    return torch.from_numpy(rs.standard_normal(shape).astype(np.float32) * by).bfloat16().to(DEV)


def _crc(t):
    return zlib.crc32(t.contiguous().cpu().view(torch.uint8).numpy().tobytes())


# the bits of a wave a row (up to 1024 rows of up to 8 times 512) and of 256
# threads, as the kernels of that form gave them
@pytest.mark.parametrize(
    "T,H,plain,added",
    [
        (300, 4096, 1155317914, 3384798846),
        (256, 3584, 1875087162, 4232488449),
        (1024, 2560, 2068124969, 3448840648),
        (1024, 2048, 2901111737, 1074708348),
        (1100, 4096, 2573155173, 615605886),
        (512, 8192, 3952354141, 3627967014),
        (700, 3584, 1197349832, 870466643),
    ],
)
def test_rmsnorm_order(T, H, plain, added):
    rs = np.random.RandomState(T + H)
    x, r = (_rows(rs, T, H, by=2) for _ in range(2))
    w = _rows(rs, H)
    assert _crc(ops.rmsnorm(x, w, 1e-5)) == plain
    assert _crc(ops.rmsnorm_residual(x, r, w, 1e-5)[0]) == added


# every split of K that the fragment-major kernel has, row tiles of 64 to 256
@pytest.mark.parametrize("M", [9, 16, 40, 64, 65, 128, 129, 256])
@pytest.mark.parametrize(
    "N,K", [(4096, 4096), (4096, 8256), (3584, 3584), (2048, 1024), (8192, 8192), (8192, 8256),
            (7168, 2048), (64, 2048)])
def test_linear_in_order(M, N, K):
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * K**-0.5).bfloat16()
    cfg = ops._m256_config(M, N, K)
    got = ops.linear_in_order(x, w)
    if cfg is None:
        want = ops._linear_slabs(x, w)
    else:
        want = ops.gemm_m256(x, ops.swizzle_weight_frag(w), **cfg)
        assert torch.equal(ops.linear_in_order(x, w, ops.swizzle_weight_frag(w)), want)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M", [9, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("N", [28672, 7168])
def test_swiglu_linear_in_order(M, N, K=4096):
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=DEV).bfloat16()
    w = (torch.randn(N, K, device=DEV) * K**-0.5).bfloat16()
    twin = ops.swizzle_weight_frag(ops.interleave_gate_up(w))
    want = ops.gemm_m256_swiglu(x, twin, **ops._m256_swiglu_config(M, N, K))
    assert torch.equal(ops.swiglu_linear_in_order(x, w), want)
    assert torch.equal(ops.swiglu_linear_in_order(x, w, w_int=twin), want)


def test_sum_parts_refuses():
    parts = torch.zeros(2, 4, 64, device=DEV)
    y = torch.zeros(4, 64, device=DEV).bfloat16()
    for args in ((y[:3], parts), (y, parts.double()), (y, parts[0]), (y[:, :32], parts)):
        with pytest.raises(RuntimeError):
            ops._native().sum_parts(*args)
