"""Op dispatch: gfx950 HIP kernels on GPU, PyTorch reference on CPU.

The HIP extensions (llmapigateway_amd/ops/_C*.so and _H*.so, built in-tree by
``python setup.py build_ext --inplace`` / __graft_entry__.build; see native.py)
are the ONLY compute path on GPU tensors — if a CUDA tensor reaches an op and
its extension is missing, we raise instead of silently falling back to eager
PyTorch. CPU tensors use ops.reference (fp32 semantics contract).
"""

from __future__ import annotations

import os
from typing import Optional, Tuple

# Enable the pre-tuned hipBLASLt/rocBLAS GEMM selections for gfx950 (3.2x on
# the decode lm_head GEMM). torch appends the device ordinal before ".csv",
# so the shipped table is tunableop_gfx950<N>.csv and FILENAME names the
# base. Must be set before the first GEMM executes; honor user overrides.
_TUNE_BASE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tunableop_gfx950.csv")
if os.path.exists(_TUNE_BASE.replace(".csv", "0.csv")):
    os.environ.setdefault("PYTORCH_TUNABLEOP_ENABLED", "1")
    os.environ.setdefault("PYTORCH_TUNABLEOP_TUNING", "0")
    os.environ.setdefault("PYTORCH_TUNABLEOP_FILENAME", _TUNE_BASE)

import torch

# Belt-and-braces: activate TunableOp through the python API too (the env
# vars alone were not picked up when torch was imported first elsewhere).
if torch.version.hip and os.path.exists(_TUNE_BASE.replace(".csv", "0.csv")):
    try:
        import torch.cuda.tunable as _tunable

        _tunable.enable(True)
        # honor an explicit tuning request (tools/tune_gemms.py sets "1");
        # otherwise lock to lookup-only so serving never pays tuning cost
        if os.environ.get("PYTORCH_TUNABLEOP_TUNING") != "1":
            _tunable.tuning_enable(False)
            _tunable.set_filename(_TUNE_BASE, insert_device_ordinal=True)
            _tunable.read_file(_TUNE_BASE.replace(".csv", "0.csv"))
    except Exception:  # pragma: no cover - best effort
        pass

from . import reference
from .reference import build_rope_cache  # re-export (host-side table builder)

from .native import dense_native as _native, have_native, shared_native as _shared


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().rmsnorm(out, x, weight, eps)
        return out
    return reference.rmsnorm(x, weight, eps)


def rmsnorm_residual(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5
) -> Tuple[torch.Tensor, torch.Tensor]:
    if x.is_cuda:
        # fused: residual += x; x_out = rmsnorm(residual) — one HBM pass
        out = torch.empty_like(x)
        _native().rmsnorm_residual(out, x, residual, weight, eps)
        return out, residual
    return reference.rmsnorm_residual(x, residual, weight, eps)


def rope_inplace(
    q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor
) -> None:
    if q.is_cuda:
        _native().rope_inplace(q, k, positions, cos_sin)
        return
    reference.rope_inplace(q, k, positions, cos_sin)


def swiglu(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        inter = x.shape[-1] // 2
        out = torch.empty(
            (*x.shape[:-1], inter), dtype=x.dtype, device=x.device
        )
        _shared().swiglu(out, x)
        return out
    return reference.swiglu(x)


def rope_and_kv_write(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    positions: torch.Tensor,
    cos_sin: torch.Tensor,
    slot_mapping: torch.Tensor,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
) -> None:
    """Fused rope_inplace(q, k) + kv_cache_write(k, v): one launch on GPU.
    With k_scale/v_scale the cache is fp8 e4m3 (per-row quantization)."""
    if q.is_cuda:
        _native().rope_kv_write(
            q, k, v, k_cache, v_cache, positions, cos_sin, slot_mapping,
            k_scale, v_scale,
        )
        return
    reference.rope_inplace(q, k, positions, cos_sin)
    reference.kv_cache_write(k, v, k_cache, v_cache, slot_mapping, k_scale, v_scale)


def kv_cache_write(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
) -> None:
    if k.is_cuda:
        _native().kv_cache_write(k, v, k_cache, v_cache, slot_mapping, k_scale, v_scale)
        return
    reference.kv_cache_write(k, v, k_cache, v_cache, slot_mapping, k_scale, v_scale)


QTILE = 64  # q rows per prefill workgroup (must match attention_prefill.hip)


def build_prefill_tiles(seqlens, device) -> Tuple[torch.Tensor, torch.Tensor]:
    """Host-side tile map for the prefill kernel: one entry per 64-row q tile."""
    tile_seq, tile_off = [], []
    for i, L in enumerate(seqlens):
        for off in range(0, int(L), QTILE):
            tile_seq.append(i)
            tile_off.append(off)
    return (
        torch.tensor(tile_seq, dtype=torch.int32, device=device),
        torch.tensor(tile_off, dtype=torch.int32, device=device),
    )


def attention_prefill(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    cu_seqlens: torch.Tensor,
    max_seqlen: int,
    scale: Optional[float] = None,
    causal: bool = True,
    tile_seq: Optional[torch.Tensor] = None,
    tile_off: Optional[torch.Tensor] = None,
    k_cache: Optional[torch.Tensor] = None,
    v_cache: Optional[torch.Tensor] = None,
    block_tables: Optional[torch.Tensor] = None,
    cached_lens: Optional[torch.Tensor] = None,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """Varlen causal prefill. With cached_lens set, each sequence also
    attends (unmasked) to its first cached_lens[i] positions read from the
    paged KV cache via block_tables — the prefix-caching / chunked-prefill
    context phase."""
    if scale is None:
        scale = float(q.shape[-1]) ** -0.5
    if q.is_cuda:
        if not causal:
            raise NotImplementedError("GPU prefill kernel is causal-only")
        if tile_seq is None or tile_off is None:
            cu = cu_seqlens.cpu().tolist()
            seqlens = [cu[i + 1] - cu[i] for i in range(len(cu) - 1)]
            tile_seq, tile_off = build_prefill_tiles(seqlens, q.device)
        out = torch.empty_like(q)
        _native().attention_prefill(
            out, q, k, v, cu_seqlens.int(), tile_seq, tile_off, float(scale),
            k_cache, v_cache, block_tables, cached_lens, k_scale, v_scale,
        )
        return out
    return reference.attention_prefill(
        q, k, v, cu_seqlens, scale, causal,
        k_cache=k_cache, v_cache=v_cache,
        block_tables=block_tables, cached_lens=cached_lens,
        k_scale=k_scale, v_scale=v_scale,
    )


# the last argument of the binding, which has one kernel for every value now
_DECODE_VER = 2


def _decode_splits(pairs: int, max_context: int) -> int:
    """Spans that a context is cut into at most, by what a captured graph
    fixes: (sequence, kv head) pairs and the longest context that the tables
    hold. A workgroup streams 37 GB/s, so 168 of them already ask for what
    the memory gives, and a split costs 3 us for adding up: with 180 pairs of
    450-900 keys one span takes 16.7 us and three 19.8; below, up to 256
    workgroups (one a CU): 24 pairs of 3900-7801 keys take 34.5 us in 3 spans
    and 21 in 11; 8 pairs of 8000 keys 17.9 in 8 and 12.5 in 32."""
    if pairs >= 168:
        return 1
    return max(1, min(-(-256 // pairs), max_context // 64, 32))


def attention_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    scale: Optional[float] = None,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    if scale is None:
        scale = float(q.shape[-1]) ** -0.5
    if q.is_cuda:
        out = torch.empty_like(q)
        B, Hq, D = q.shape
        nsplit = _decode_splits(
            B * k_cache.shape[1], block_tables.shape[1] * k_cache.shape[2]
        )
        acc = ml = None
        if nsplit > 1:
            acc = torch.empty(B * Hq * nsplit * D, dtype=torch.float32, device=q.device)
            ml = torch.empty(B * Hq * nsplit * 2, dtype=torch.float32, device=q.device)
        _native().attention_decode(
            out, q, k_cache, v_cache, block_tables, context_lens, float(scale),
            acc, ml, nsplit, k_scale, v_scale, _DECODE_VER,
        )
        return out
    return reference.attention_decode(
        q, k_cache, v_cache, block_tables, context_lens, scale,
        k_scale=k_scale, v_scale=v_scale,
    )


# gemm_skinny's rows on plain weights: what gemm_stream does not take (unaligned
# operands, or more rows by SKINNY_GEMM_MAX_M).
# The 8-wave MF=2 depth-4 pipeline ties the tuned library when W is
# L3-resident (tools/gemm_probe.py rotates too little data for >100 MB
# weights, so its M>=64 rows are L3-warm and misled an M<=256 dispatch:
# in-engine, where the 16 GB weight cycle is always L3-cold, batch-256
# decode dropped 272 -> 129 req/s). In the true cold regime the library
# keeps winning at M >= 64; the custom kernel stays dispatched for the
# latency regime only.
_SKINNY_MAX_M = int(os.environ.get("SKINNY_GEMM_MAX_M", "16"))
_SKINNY_MAX_N = 28672
# per-device split-K fp32 slab scratch — each workgroup fully overwrites
# its slab stripe, so no zeroing is needed and the address is stable
# across hipGraph replays.
_skinny_ws: dict = {}


def _skinny_nsk(N: int, K: int) -> int:
    """Split-K factor: target exactly 256 workgroups (one 8-wave WG fills
    a CU; extra WGs only queue) — more splits just multiply the fp32 slab
    traffic, which at the old 512-WG target added ~60% to the weight
    stream and halved in-engine decode throughput."""
    tiles = N // 64
    nsk = max(1, -(-256 // tiles))
    nsk = min(nsk, max(1, (K // 32) // 8), 8)
    return nsk


_skinny_ws_retired: list = []  # keep old slabs alive for captured graphs


def _skinny_scratch(device, numel: int):
    ws = _skinny_ws.get(device.index)
    if ws is None or ws.numel() < numel:
        if ws is not None:
            _skinny_ws_retired.append(ws)  # a hipGraph may still replay into it
        ws = torch.empty(numel, dtype=torch.float32, device=device)
        _skinny_ws[device.index] = ws
    return ws


def swizzle_weight(w: torch.Tensor) -> torch.Tensor:
    """[N, K] -> k-major [K/32, N, 32] for gemm_skinny's contiguous
    B-tile streams (one 4 KB block per 64-row n-stripe per k-step)."""
    N, K = w.shape
    assert K % 32 == 0 and N % 64 == 0
    return w.view(N, K // 32, 32).permute(1, 0, 2).contiguous()


def swizzle_weight_frag(w: torch.Tensor) -> torch.Tensor:
    """[N, K] -> fragment-major [K/32, N/16, 64, 8] for gemm_m256.

    Element [k32][n16][lane][e] = W[n16*16 + (lane&15)][k32*32 + (lane>>4)*8
    + e]: each 1 KiB row is exactly one wave's mfma_f32_16x16x32_bf16
    B-fragment in lane order, so the kernel's global_load_lds staging is a
    straight contiguous copy and its ds_read_b128 is lane-linear
    (conflict-free per the gfx950 b128 lane groups)."""
    N, K = w.shape
    assert K % 64 == 0 and N % 64 == 0
    return (
        w.view(N // 16, 16, K // 32, 4, 8)
        .permute(2, 0, 3, 1, 4)
        .reshape(K // 32, N // 16, 64, 8)
        .contiguous()
    )


def _m256_config(M: int, N: int, K: int) -> Optional[dict]:
    """Measured dispatch table for the decode projections (cold-L3 sweep,
    profiles/r02_gemm_m256_sweep.md). Returns gemm_m256 kwargs, or None
    when the tuned library wins the shape (gate_up N=28672, lm_head)."""
    if M > 256:
        return None
    if N == 8192 and K % 64 == 0 and K >= 8192:
        # 70B-class projections at tp=1 (hidden 8192): o-proj K=8192
        # (51.2 vs library 58.2 us) and down-proj K=28672 (147.5 vs
        # 192.4 us) — register-staged variant wins the deep-K shape
        if K > 8192:
            return {"nf": 8, "nsk": 4, "variant": 1, "pipe": 0}  # 70B down 1.30x
        return {"nf": 8, "nsk": 4, "variant": 0, "pipe": 0}      # 70B o 1.14x
    if N == 7168 and K <= 8192:
        # tp=4 gate_up shard (unfused path): 37.3 vs library 43.4 us
        return {"nf": 4, "nsk": 3, "variant": 0, "pipe": 4}
    if N > 4096:
        # library wins the very wide shapes: gate_up N=28672/57344
        # (custom best 73.3 vs 70.3 us / 287.9 vs 258.0), qkv N=6144
        # (36.4 vs ~28 us — hipBLASLt's MT112x256 kernel is strong
        # exactly there) and N=10240 (77.7 vs 66.7), lm_head
        return None
    if K > 8192 and N % 128 == 0:
        return {"nf": 8, "nsk": 8, "variant": 0, "pipe": 0}  # down 1.34x
    if N < 2048:
        # narrow column shards (tp=4 qkv N=1536): too few tiles to fill
        # the chip — library 1.8x faster (21.7 vs 39.7 us)
        return None
    if K < 2048:
        # shallow-K row shards (tp=4 o-proj K=1024): single-pass
        # register-staged wins 1.67x (12.7 vs 21.2 us); split-K slab
        # traffic would dominate this little work
        return {"nf": 4, "nsk": 1, "variant": 1, "pipe": 0}
    # o-proj class (N<=4096, K<=8192): BK64/NBUF2 2-blocks/CU + split-K
    tiles = N // 64
    nsk = max(1, min(-(-256 // tiles), (K // 64) // 2, 8))
    return {"nf": 4, "nsk": nsk, "variant": 0, "pipe": 4}  # o 1.30x


def _m256_nsk(N: int, K: int, nf: int) -> int:
    """Split-K factor for gemm_m256: fill the 256 CUs (one 8-wave block
    per CU at the 120 KB LDS ring) when the column-tile count alone
    cannot. The fp32 slab traffic (2*nsk*M*N*4 B) is the price, so tiles
    >= 256 never split; smaller-N shapes are load-path/latency-bound and
    the slab round trip is cheap relative to the CU-fill win
    (profiles/r02_gemm_m256_probe.md)."""
    tiles = N // (16 * nf)
    if tiles >= 256:
        return 1
    nsk = -(-256 // tiles)
    return max(1, min(nsk, (K // 64) // 2, 8))


# swizzled weights raise the profitable dispatch ceiling (contiguous
# streams); plain-layout dispatch stays in the latency regime
_SKINNY_SWZ_MAX_M = int(os.environ.get("SKINNY_GEMM_SWZ_MAX_M", "256"))


# 0 = glds-staged, 1 = register-staged T14 (see gemm_m256.hip header)
_M256_VARIANT = int(os.environ.get("LLMAPI_M256_VARIANT", "0"))


def gemm_m256(
    x: torch.Tensor, w_frag: torch.Tensor, nf: Optional[int] = None,
    nsk: Optional[int] = None, variant: Optional[int] = None,
    pipe: Optional[int] = None,
) -> torch.Tensor:
    """y = x @ w.T with w pre-swizzled fragment-major (swizzle_weight_frag).
    The macro-tile LDS-staged decode GEMM (csrc/gemm_m256.hip); M <= 256.
    pipe selects the DMA ring geometry for the glds variant:
    0=(BK64,N3) 1=(BK64,N4,nf4) 2=(BK32,N4,nf8) 3=(BK32,N6,nf8)."""
    M, K = x.shape
    N = w_frag.shape[1] * 16
    if nf is None:
        if N % 128 == 0 and M > 64:
            nf = 8  # deep BK32 ring needs BN=128
        else:
            nf = 8 if N // 64 >= 448 else 4
    if N % (16 * nf) != 0:
        nf = 4
    if nsk is None:
        nsk = _m256_nsk(N, K, nf)
    if variant is None:
        variant = _M256_VARIANT
    if pipe is None:
        pipe = 3 if (variant == 0 and nf == 8 and K % 32 == 0) else 0
    if variant == 0:
        if pipe in (2, 3) and nf != 8:
            pipe = 0
        if pipe in (1, 4, 5) and nf != 4:
            pipe = 0
    y = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
    ws = _skinny_scratch(x.device, nsk * M * N) if nsk > 1 else None
    _native().gemm_m256(y, x, w_frag, ws, nsk, nf, variant, pipe, 0)
    return y


def interleave_gate_up(w: torch.Tensor) -> torch.Tensor:
    """Row-permute a [gate; up] stacked weight [2I, K] into block-16
    interleaved order [g0..15, u0..15, g16..31, ...]: after
    swizzle_weight_frag, the gate/up accumulators for the same output
    column land in the SAME lane of adjacent 16-col fragments, which is
    what gemm_m256's fused swiglu epilogue consumes."""
    two_i, K = w.shape
    assert two_i % 32 == 0
    return w.view(2, two_i // 32, 16, K).transpose(0, 1).reshape(two_i, K)


def gemm_m256_swiglu(
    x: torch.Tensor, w_frag: torch.Tensor, nf: int = 8, variant: int = 1,
    pipe: int = 0,
) -> torch.Tensor:
    """silu(x @ gate.T) * (x @ up.T) in ONE kernel: w_frag is
    swizzle_weight_frag(interleave_gate_up(gate_up)) and the swiglu runs
    in the GEMM epilogue on the fp32 accumulators — the [M, 2I]
    intermediate round trip and the separate swiglu kernel disappear
    (~72 MB of HBM traffic per llama-3-8b layer at M=256)."""
    M, K = x.shape
    N = w_frag.shape[1] * 16
    y = torch.empty((M, N // 2), dtype=torch.bfloat16, device=x.device)
    _native().gemm_m256(y, x, w_frag, None, 1, nf, variant, pipe, 1)
    return y


def _m256_swiglu_config(M: int, N: int, K: int) -> Optional[dict]:
    """Measured dispatch for the FUSED gate_up+swiglu decode MLP front
    (profiles/r02_gemm_m256_sweep.md). N is the stacked 2*intermediate.
    Only the 8B shape measured ahead of library+swiglu (77.2 vs 79.4 us
    cold-L3); the 70B shape loses (304.8 vs 226.6) and stays unfused."""
    if os.environ.get("LLMAPI_NO_FUSED_SWIGLU"):
        return None
    if not (8 < M <= 256):
        return None
    if N == 28672 and K == 4096:  # llama-3-8b tp=1
        if M <= 128:  # 55.0 vs 61.8 us at M=128 (glds variant)
            return {"nf": 8, "variant": 0, "pipe": 0}
        return {"nf": 8, "variant": 1, "pipe": 0}
    if N == 7168 and K == 4096:  # tp=4 gate_up shard: 45.9 vs 46.8 us
        return {"nf": 4, "variant": 0, "pipe": 4}
    return None


def _streams(M: int, N: int, K: int) -> bool:
    """Whether gemm_stream takes a product: it reads W at the memory's rate
    without a second kernel, but every 16 columns read all rows of x. Up to 16
    rows it beats the library and the slab kernel at every width (4096 x 4096:
    8.5 us, 11-15 before; 6144 x 4096: 13.4, 19.8) except that of a head, where
    the rows' part shows (128256 x 4096: 155 us at one row where the library
    takes 158, 187 at 16 where it takes 185). Beyond, it wins where columns are
    few (32 rows, 4096 x 14336: 30 us, macro tile 38; 64 rows, 4096 x 4096: 13.8
    and 14.5, 4096 x 14336: 44 and 32)."""
    if M <= 16:
        return M <= 8 or N <= 65536
    return N <= 4096 and (M <= 32 or (M <= 64 and K <= 4096))


def _streams_swiglu(M: int, N: int) -> bool:
    """The same with swiglu behind it, N the stacked width: 28672 x 4096 takes
    40-41 us up to 16 rows (54-66 before), 46 at 32 (66), 53 at 48 (54). Up to 16
    rows at 57344 x 8192 both are at the memory's rate (171 and 166). Beyond,
    workgroups have 64 columns: too few of them below 16384 (7168 x 4096 at 32
    rows: 22 us, library and swiglu 19.5), and above 32 rows two rounds of them
    over 32768 (37888 x 3584 at 48 rows: 72 and 64); small ones are launches
    (1024 x 512: 4.7 and 8)."""
    if M <= 16:
        return N <= 40960
    if M <= 48:
        return N <= 4096 or 16384 <= N <= (40960 if M <= 32 else 32768)
    return False


def _streamable(x: torch.Tensor, w: torch.Tensor) -> bool:
    """What gemm_stream asks of its operands; it has no derivative."""
    return (
        x.is_cuda and x.dim() == 2 and x.shape[0] > 0
        and w.numel() > 0 and w.shape[1] < 2**25
        and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
        and not ((x.requires_grad or w.requires_grad) and torch.is_grad_enabled())
        and x.is_contiguous() and w.is_contiguous()
        and w.shape[0] % 64 == 0 and w.shape[1] % 32 == 0
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
    )


def swiglu_linear(
    x: torch.Tensor, w: torch.Tensor,
    w_swz: Optional[torch.Tensor] = None,
    w_int: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """MLP front: swiglu(x @ w.T) with w = [gate; up] stacked. Few rows go
    to gemm_stream; others to the fused gemm_m256 epilogue when the
    interleaved twin exists and the measured table says it wins; otherwise
    library GEMM + swiglu kernel."""
    if (
        _streamable(x, w) and _streams_swiglu(x.shape[0], w.shape[0])
        and not os.environ.get("LLMAPI_NO_FUSED_SWIGLU")
    ):
        y = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype, device=x.device)
        _shared().gemm_stream(y, x, w, True)
        return y
    if w_int is not None and x.dim() == 2:
        cfg = _m256_swiglu_config(x.shape[0], w_int.shape[1] * 16, x.shape[1])
        if cfg is not None:
            return gemm_m256_swiglu(x, w_int, **cfg)
    return swiglu(linear(x, w, w_swz))


def linear(
    x: torch.Tensor, w: torch.Tensor, w_swz: Optional[torch.Tensor] = None
) -> torch.Tensor:
    """y = x @ w.T. bf16 products of few rows stream the weight
    (csrc/gemm_stream.hip); other decode-shaped ones (M <= 256) go through the
    macro-tile gfx950 kernel (csrc/gemm_m256.hip) when the fragment-major
    weight twin exists (models/llama.py builds them); everything else
    through the TunableOp-tuned library GEMMs."""
    M = x.shape[0]
    if (w_swz is None or w_swz.dim() == 4) and _streamable(x, w) and _streams(M, *w.shape):
        y = torch.empty((M, w.shape[0]), dtype=torch.bfloat16, device=x.device)
        _shared().gemm_stream(y, x, w, False)
        return y
    return _linear_slabs(x, w, w_swz)


def _linear_slabs(
    x: torch.Tensor, w: torch.Tensor, w_swz: Optional[torch.Tensor] = None
) -> torch.Tensor:
    M = x.shape[0]
    if (
        x.is_cuda
        and x.dtype == torch.bfloat16
        and w.dtype == torch.bfloat16
        and 0 < M
        and w.shape[0] % 64 == 0
        and w.shape[0] <= _SKINNY_MAX_N
        and w.shape[1] % 32 == 0
        and x.is_contiguous()
        and w.is_contiguous()
    ):
        N, K = w.shape
        if (
            w_swz is not None
            and w_swz.dim() == 4
            and 8 < M <= 256
            and K % 64 == 0
        ):
            cfg = _m256_config(M, N, K)
            if cfg is not None:
                return gemm_m256(x, w_swz, **cfg)
            # fall through to library (measured faster for this shape)
            return torch.nn.functional.linear(x, w)
        if w_swz is not None and w_swz.dim() == 3 and M <= _SKINNY_SWZ_MAX_M:
            # legacy k-major twin -> streaming skinny kernel
            y = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
            nsk = _skinny_nsk(N, K)
            ws = _skinny_scratch(x.device, nsk * M * N) if nsk > 1 else None
            _shared().gemm_skinny(y, x, w_swz, ws, nsk, True)
            return y
        if M <= _SKINNY_MAX_M:
            y = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
            nsk = _skinny_nsk(N, K)
            ws = _skinny_scratch(x.device, nsk * M * N) if nsk > 1 else None
            _shared().gemm_skinny(y, x, w, ws, nsk, False)
            return y
    return torch.nn.functional.linear(x, w)


# ---- a prompt's products in an order that does not change ----
# What a prompt leaves in pages of e4m3 is bytes: a sum in another order turns
# none of bf16's digits that count, but moves a quarter of the codes after four
# layers. So the rows of a prompt have their sums where they have always been:
# up to 16 by gemm_skinny, up to 256 as gemm_m256 sums (from the weight as it
# lies: gemm_tile in the same splits of K), others by the library.


def linear_in_order(
    x: torch.Tensor, w: torch.Tensor, w_swz: Optional[torch.Tensor] = None,
    head: bool = False,
) -> torch.Tensor:
    """linear() of one of a layer's weights, in the order that a fragment-major
    twin gives, whether there is one or not; heads have none."""
    if w_swz is None and not head and x.is_cuda and 8 < x.shape[0] <= 256 and _twin_fits(w):
        (M, K), N = x.shape, w.shape[0]
        cfg = _m256_config(M, N, K)
        if cfg is not None and _streamable(x, w):
            parts = torch.empty((cfg["nsk"], M, N), dtype=torch.float32, device=x.device)
            _native().gemm_tile(parts, x, w, True)
            y = torch.empty((M, N), dtype=x.dtype, device=x.device)
            _native().sum_parts(y, parts)
            return y
    return _linear_slabs(x, w, w_swz)


def _twin_fits(w: torch.Tensor) -> bool:
    return _tileable(w) and w.shape[0] % 64 == 0 and not os.environ.get("LLMAPI_NO_FRAG_WEIGHTS")


def swiglu_linear_in_order(
    x: torch.Tensor, w: torch.Tensor,
    w_swz: Optional[torch.Tensor] = None,
    w_int: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """swiglu_linear() in the same way."""
    cfg = _m256_swiglu_config(x.shape[0], *w.shape) if x.is_cuda else None
    if cfg is not None and w_int is not None:
        return gemm_m256_swiglu(x, w_int, **cfg)
    if cfg is not None and _twin_fits(w) and _streamable(x, w):
        y = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype, device=x.device)
        _native().gemm_tile(y, x, w, True)
        return y
    return swiglu(linear_in_order(x, w, w_swz))


# ---- a decode step's products with what stands beside them ----
# The stream r is the layer's input plus every sublayer's output, [T, hidden].
# Few rows have each sublayer in two products (csrc/gemm_stream.hip).


def layer_streams(T: int, layer: dict) -> bool:
    """Whether a layer's four products all go to gemm_stream with their norms,
    additions and rotation: 4 launches instead of 10 or 13. Above 16 rows tiles
    are ahead for large layers (32 rows of hidden size 4096: 110 us a layer
    streamed, 105 tiled; of 3584: 120 and 109), for smaller ones the fewer
    launches (3072: 60 and 66; 2048: 43 and 44)."""
    if not 0 < T <= 32:
        return False
    qkv, o, gate_up, down = weights = [layer[k] for k in ("qkv", "o", "gate_up", "down")]
    return (
        (T <= 16 or gate_up.numel() < 2**26)
        and all(
            w.is_cuda and w.dtype == torch.bfloat16 and w.is_contiguous()
            and w.shape[0] % 64 == 0 and w.shape[1] % 32 == 0 and w.data_ptr() % 16 == 0
            for w in weights
        )
        and not any(k.endswith("_swz") and w.dim() == 3 for k, w in layer.items())
        and _streams(T, *o.shape) and _streams(T, *down.shape)
        and qkv.shape[0] <= (65536 if T <= 16 else 12288)
        and _streams_swiglu(T, gate_up.shape[0])
    )


def embed_rows(
    tokens: torch.Tensor, embed: torch.Tensor, norm: torch.Tensor, eps: float,
    normed: bool = True,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """The tokens' rows of embed, and their RMS norm if asked for."""
    if (
        embed.is_cuda and embed.dtype == torch.bfloat16 and embed.is_contiguous()
        and embed.data_ptr() % 16 == 0 and tokens.numel() > 0 and tokens.dim() == 1
        and tokens.dtype == torch.long and tokens.is_contiguous()
        and embed.shape[1] % 8 == 0 and embed.shape[1] <= 16384  # what a workgroup holds
    ):
        r = torch.empty(
            (tokens.shape[0], embed.shape[1]), dtype=embed.dtype, device=embed.device
        )
        x = torch.empty_like(r) if normed else None
        _native().embed_norm(x, r, tokens, embed, norm, eps)
        return r, x
    r = torch.nn.functional.embedding(tokens, embed)
    return r, rmsnorm(r, norm, eps) if normed else None


def norm_qkv_rotated(
    r: torch.Tensor, norm: torch.Tensor, eps: float, w: torch.Tensor,
    positions: torch.Tensor, cos_sin: torch.Tensor, slots: torch.Tensor,
    k_cache: torch.Tensor, v_cache: torch.Tensor,
    k_scale: Optional[torch.Tensor] = None, v_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """rmsnorm(r) @ w.T as rows of query, key and value heads, the first two
    rotated; keys and values are also written to their pages."""
    if r.is_cuda:
        y = torch.empty((r.shape[0], w.shape[0]), dtype=r.dtype, device=r.device)
        if k_scale is not None:  # a scale needs all of a row: a kernel of its own
            if r.shape[0] <= 16:
                _native().gemm_stream_rows(y, r, w, 0, norm, eps)
            else:
                y = linear(rmsnorm(r, norm, eps), w)
            Hkv, D = k_cache.shape[1], k_cache.shape[3]
            heads = y.view(r.shape[0], -1, D)
            q, k, v = heads.split([heads.shape[1] - 2 * Hkv, Hkv, Hkv], dim=1)
            rope_and_kv_write(
                q, k, v, k_cache, v_cache, positions, cos_sin, slots,
                k_scale=k_scale, v_scale=v_scale,
            )
            return y
        _native().gemm_stream_qkv(
            y, r, w, norm, eps, positions, cos_sin, slots, k_cache, v_cache
        )
        return y
    y = reference.rmsnorm(r, norm, eps) @ w.T
    return _rotated_(y, positions, cos_sin, slots, k_cache, v_cache, k_scale, v_scale)


def _rotated_(y, positions, cos_sin, slots, k_cache, v_cache, k_scale, v_scale):
    Hkv, D = k_cache.shape[1], k_cache.shape[3]
    heads = y.view(y.shape[0], -1, D)
    q, k, v = heads.split([heads.shape[1] - 2 * Hkv, Hkv, Hkv], dim=1)
    reference.rope_inplace(q, k, positions, cos_sin)
    kept = slots >= 0
    reference.kv_cache_write(
        k[kept], v[kept], k_cache, v_cache, slots[kept], k_scale, v_scale
    )
    return y


def norm_swiglu_linear(
    r: torch.Tensor, norm: torch.Tensor, eps: float, w: torch.Tensor
) -> torch.Tensor:
    """swiglu(rmsnorm(r) @ w.T), w = [gate; up] stacked."""
    if r.is_cuda and os.environ.get("LLMAPI_NO_FUSED_SWIGLU"):
        return swiglu(linear(rmsnorm(r, norm, eps), w))
    if r.is_cuda:
        y = torch.empty((r.shape[0], w.shape[0] // 2), dtype=r.dtype, device=r.device)
        _native().gemm_stream_rows(y, r, w, 1, norm, eps)
        return y
    return reference.swiglu(reference.rmsnorm(r, norm, eps) @ w.T)


def linear_add_(x: torch.Tensor, w: torch.Tensor, r: torch.Tensor) -> torch.Tensor:
    """r += x @ w.T"""
    if r.is_cuda:
        _native().gemm_stream_rows(r, x, w, 2, None, 0.0)
        return r
    return r.add_(x @ w.T)


def norm_logits(
    r: torch.Tensor, norm: torch.Tensor, eps: float, w: torch.Tensor
) -> torch.Tensor:
    """rmsnorm(r) @ w.T in fp32."""
    return logits_linear(rmsnorm(r, norm, eps) if r.shape[0] else r, w)


# A batch's rows have the products in tiles (csrc/gemm_tile.hip), K split over
# workgroups; what reads the parts adds them up (csrc/parts_rows.hip).


def _tileable(w: torch.Tensor) -> bool:
    return (
        w.is_cuda and w.dtype == torch.bfloat16 and w.is_contiguous()
        and w.shape[0] % 32 == 0 and w.shape[1] % 64 == 0 and w.numel() < 2**31
        and w.data_ptr() % 16 == 0
    )


def layer_tiles(T: int, layer: dict, head_dim: int) -> bool:
    """Whether a layer of T rows, not streamed, goes to gemm_tile: 7 launches
    instead of 11 to 14. Layers of hidden size 2048 gain at every number of rows
    (48 rows: 45 us, 51.5 before; 256: 77 and 89), of 1024 up to 128 (48: 32 and
    34.5; 128: 36 and 41; 200: 51 and 48), of 512 lose (48: 27 and 24). Up to 8
    rows a large layer gains (8192: 325 and 348 at one row), others do not (3072
    in products of few rows and small kernels: 61 at 16 rows, 62 in tiles). Above
    256 rows single products do."""
    hidden = layer["qkv"].shape[1]
    return (
        (8 if hidden < 8192 else 0) < T <= 512 and head_dim == 128
        and (1024 if T <= 128 else 2048) <= hidden <= 16384  # what add_parts_norm holds
        and all(_tileable(layer[k]) for k in ("qkv", "o", "gate_up", "down"))
        and not any(k.endswith("_swz") and w.dim() == 3 for k, w in layer.items())
    )


def _parts_pay(M: int, N: int) -> bool:
    """Whether a product of a tiled layer comes in parts: up to 256 rows all, up
    to 512 those of few columns (300 rows: 4096 x 4096 with its addition and norm
    28 us, library 30, 4096 x 14336 74 and 76, 3584 x 18944 82 and 102, with
    rotation 4608 x 3584 27 and 30, but 6144 x 4096 44 and 37; 512 rows: 32 and
    33.5, 83 and 91, 82 and 201, 42 and 40, 51 and 49)."""
    return M <= 256 or N <= (4608 if M <= 448 else 4096)


def linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w.T in fp32 as parts to be added up, [parts, T, N]."""
    if x.is_cuda:
        (M, K), N = x.shape, w.shape[0]
        splits = _native().gemm_tile_splits(M, N, K)
        y = torch.empty((splits, M, N), dtype=torch.float32, device=x.device)
        _native().gemm_tile(y, x, w)
        return y
    return (x.float() @ w.float().T)[None]


def rotated_parts(
    parts: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor, slots: torch.Tensor,
    k_cache: torch.Tensor, v_cache: torch.Tensor, dtype: torch.dtype = torch.bfloat16,
    k_scale: Optional[torch.Tensor] = None, v_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """The sum of parts as rows of query, key and value heads, the first two
    rotated; keys and values are also written to their pages."""
    if parts.is_cuda:
        y = torch.empty(parts.shape[1:], dtype=dtype, device=parts.device)
        _native().rotate_parts(
            y, parts, positions, cos_sin, slots, k_cache, v_cache, k_scale, v_scale
        )
        return y
    return _rotated_(
        parts.sum(0).to(dtype), positions, cos_sin, slots, k_cache, v_cache, k_scale, v_scale
    )


def add_parts_norm_(
    r: torch.Tensor, parts: torch.Tensor, norm: torch.Tensor, eps: float
) -> torch.Tensor:
    """r += the sum of parts; returns rmsnorm(r)."""
    if r.is_cuda:
        out = torch.empty_like(r)
        _native().add_parts_norm(out, r, parts, norm, eps)
        return out
    return reference.rmsnorm(r.add_(parts.sum(0).to(r.dtype)), norm, eps)


def qkv_rotated(
    x: torch.Tensor, w: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor,
    slots: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    k_scale: Optional[torch.Tensor] = None, v_scale: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """x @ w.T as rows of query, key and value heads, the first two rotated;
    keys and values are also written to their pages."""
    if _parts_pay(x.shape[0], w.shape[0]):
        return rotated_parts(
            linear_parts(x, w), positions, cos_sin, slots, k_cache, v_cache, x.dtype,
            k_scale, v_scale,
        )
    y = linear(x, w)
    Hkv, D = k_cache.shape[1], k_cache.shape[3]
    heads = y.view(x.shape[0], -1, D)
    q, k, v = heads.split([heads.shape[1] - 2 * Hkv, Hkv, Hkv], dim=1)
    rope_and_kv_write(
        q, k, v, k_cache, v_cache, positions, cos_sin, slots,
        k_scale=k_scale, v_scale=v_scale,
    )
    return y


def linear_add_norm_(
    x: torch.Tensor, w: torch.Tensor, r: torch.Tensor, norm: torch.Tensor, eps: float
) -> torch.Tensor:
    """r += x @ w.T; returns rmsnorm(r)."""
    if not r.is_cuda or _parts_pay(x.shape[0], w.shape[0]):
        return add_parts_norm_(r, linear_parts(x, w), norm, eps)
    return rmsnorm_residual(linear(x, w), r, norm, eps)[0]


def _tiles_wide(M: int, N: int, K: int) -> bool:
    """Whether a product without splits is one for gemm_tile: above 128 rows the
    library's is ahead where columns make several rounds and K is long (256 rows,
    57344 x 8192 and swiglu: 247 us, library 242; 128256 x 8192 in fp32: 506 and
    504; with K 4096: 266 and 358)."""
    return M <= 128 or (M <= 256 and (K <= 4096 or N <= 32768))


def swiglu_tiled(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """swiglu(x @ w.T), w = [gate; up] stacked."""
    if (
        x.is_cuda and _tiles_wide(x.shape[0], *w.shape)
        and not os.environ.get("LLMAPI_NO_FUSED_SWIGLU")
    ):
        y = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype, device=x.device)
        _native().gemm_tile(y, x, w)
        return y
    return swiglu(torch.nn.functional.linear(x, w))


def logits_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w.T in fp32, for a head."""
    M = x.shape[0]
    if 0 < M <= 256 and _streamable(x, w):
        y = torch.empty((M, w.shape[0]), dtype=torch.float32, device=x.device)
        if M <= 16 and _streams(M, *w.shape):
            _native().gemm_stream_rows(y, x, w, 3, None, 0.0)
            return y
        if _tileable(w) and w.shape[1] >= 1024 and _tiles_wide(M, *w.shape):
            _native().gemm_tile(y, x, w)
            return y
    return linear(x, w).float()


def topk_topp_filter(
    logits: torch.Tensor, topp: torch.Tensor, topk: torch.Tensor
) -> torch.Tensor:
    """Mask logits outside the per-row top-k / top-p set to -inf, in
    place, and return logits. GPU: histogram-threshold kernel
    (csrc/sampling.hip, no sort, no host loop); CPU: batched torch sort
    (reference semantics)."""
    if logits.is_cuda:
        _native().topk_topp_filter(logits, topp, topk)
        return logits
    return reference.topk_topp_filter(logits, topp, topk)


def sample(
    logits: torch.Tensor,
    temperature: torch.Tensor,
    noise: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.long, device=logits.device)
        _native().sample(out, logits, temperature, noise)
        return out
    return reference.sample(logits, temperature, noise)


from .experts import (  # noqa: E402
    ExpertSum, clamped_glu, expert_rows, pack_experts, route_experts,
)
from .hybrid import (  # noqa: E402
    add_cast,
    add_layernorm,
    add_rms_norm,
    add_tanh_norm,
    build_pair_rope_cache,
    can_unfold,
    causal_conv,
    decay_logs,
    decayed_kv,
    delta_kv,
    distance_bias,
    embed_rms_norm,
    embed_scaled,
    embed_tanh_norm,
    fixed_decay_kv,
    fold_queries,
    gated_norm,
    head_linear,
    head_norm_gate,
    latent_attention_folded,
    latent_attention_unfolded,
    latent_rows,
    linear_f32,
    mix_streams,
    mlstm,
    page_write,
    paged_attention,
    plan_segments,
    qkv_rows,
    rotary_rows,
    sigmoid_attention,
    soft_cap_,
    ssd,
    token_shift,
    window_attention,
    xielu_,
)

__all__ = [
    "have_native",
    "build_rope_cache",
    "rmsnorm",
    "rmsnorm_residual",
    "rope_inplace",
    "rope_and_kv_write",
    "swiglu",
    "kv_cache_write",
    "linear",
    "gemm_m256",
    "swizzle_weight",
    "swizzle_weight_frag",
    "attention_prefill",
    "attention_decode",
    "sample",
    "topk_topp_filter",
    "reference",
    "add_cast",
    "add_layernorm",
    "build_pair_rope_cache",
    "can_unfold",
    "causal_conv",
    "embed_scaled",
    "fold_queries",
    "gated_norm",
    "head_linear",
    "latent_attention_folded",
    "latent_attention_unfolded",
    "latent_rows",
    "linear_f32",
    "mlstm",
    "plan_segments",
    "ssd",
]
