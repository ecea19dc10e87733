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
