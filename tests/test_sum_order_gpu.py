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


# the last layer's pages and scales after a step over prompts of up to 16 rows
# (no library product among them), as separate kernels of slabs gave them
@pytest.mark.parametrize(
    "T,cached,bytes_,scales",
    [(5, 0, 3593197530, 1828829798), (13, 0, 315290881, 461129092),
     (16, 32, 3583420357, 2088370348)],
)
def test_prompt_bytes(T, cached, bytes_, scales):
    from llmapigateway_amd.engine.kvcache import PagedKVCache
    from llmapigateway_amd.models import build_model
    from llmapigateway_amd.models.batch import ForwardBatch
    from llmapigateway_amd.models.configs import ModelConfig

    c = ModelConfig(
        name="bytes", hidden_size=2048, intermediate_size=1024, num_layers=4, num_heads=4,
        num_kv_heads=2, vocab_size=2048, head_dim=128, rope_theta=10000.0, max_positions=1024,
    )
    model = build_model(c, device=DEV, dtype=torch.bfloat16, seed=3)
    cache = PagedKVCache(c, 8, 16, DEV, torch.bfloat16, kv_dtype="fp8")
    rs = np.random.RandomState(T)
    for pages, scale in zip(cache.k_caches + cache.v_caches, cache.k_scales + cache.v_scales):
        pages.copy_(_rows(rs, *pages.shape, by=64).float().to(torch.float8_e4m3fn).view(torch.uint8))
        scale.fill_(0.02)
    order = torch.tensor([5, 0, 7, 2], device=DEV)
    n = torch.arange(cached, cached + T, device=DEV)
    more = {}
    if cached:
        more = dict(
            block_tables=order.int().unsqueeze(0),
            cached_lens=torch.tensor([cached], dtype=torch.int32, device=DEV),
        )
    tile_seq, tile_off = ops.build_prefill_tiles([T], torch.device(DEV))
    batch = ForwardBatch(
        kind="prefill", token_ids=n * 7 % 2048, positions=n, slot_mapping=order[n // 16] * 16 + n % 16,
        cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device=DEV), max_seqlen=T,
        tile_seq=tile_seq, tile_off=tile_off,
        logits_indices=torch.tensor([T - 1], device=DEV), **more,
    )
    model.step(batch, cache)
    got = (_crc(torch.stack([cache.k_caches[-1], cache.v_caches[-1]])),
           _crc(torch.stack([cache.k_scales[-1], cache.v_scales[-1]])))
    assert got == (bytes_, scales), got
