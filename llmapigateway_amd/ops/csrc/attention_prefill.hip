// Causal prompt attention for gfx950 (MFMA bf16), varlen with GQA, over the
// step's own rows and, where a sequence has cached context (prefix caching,
// chunked prefill), over its pages in front of them.
//
// Produces the prompt phase (TTFT) the reference delegated upstream.
//
// - A workgroup has 64 query rows of up to four heads of one kv head: each wave
//   16 rows of one head, so that a key and value tile staged once serves 256
//   query columns, and 4 waves a SIMD keep its units busy (with 32 rows a wave,
//   each fragment from LDS serves two products, but 2 waves a SIMD wait for each
//   other's exponentials: 4000 tokens after 4032 512 us, 464 so; 1000 tokens 34
//   and 26).
// - S^T = K Q^T: a lane owns one query column of a block of 16, its softmax
//   state is a scalar, and the weights as they stand are the operand of
//   O^T = V^T P^T (the key order inside a product is free; V fragments come
//   from row-major tiles by transposing reads). Nothing but K and V goes
//   through LDS.
// - Tiles are transferred to LDS without registers into one of two buffers
//   while the other is in use, one barrier a tile. Pages of bytes pass through
//   registers, where they become bf16 (value times scale, rounded once).
// - Sums are in a fixed order, which no choice of workgroups touches: 64 keys at
//   a time, scores relative to the largest so far, weights as bf16 (the largest is
//   1 and loses nothing) for the values and as fp32 for their sum. What a prompt
//   leaves behind in pages of bytes so depends on the prompt alone. (A maximum
//   that moves only past 2^8 saves a tenth of the time, but rounds the largest
//   weights, too: over 4000 keys the weights' share of the error is 1.6e-3 then,
//   1.25e-3 so.)
// - Blocks of one kv head follow each other at the distance of the XCDs, and
//   late tiles, which see the most keys, start first.
//
// One layer, 32 query and 8 kv heads; before: 64 rows and one head a workgroup,
// keys and values through registers, weights through LDS:
//   4096 tokens                   1117 us -> 189 us (727 TFLOP/s)
//   4000 tokens after 4032        2371    -> 464    (852), from e4m3 pages 494
//   9 x 117-213 tokens after 1984  428    ->  87
//   32 x 66-128 tokens              46    ->  23
//   37 tokens                      6.6    -> 6.1
// Long prompts are bound by the vector ALU beside the matrix cores (an
// exponential and 6 operations a score, the sums' rescaling).

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

#define PF_D 128
#define QTILE 64  // query rows of a tile (ops.build_prefill_tiles)
#define PF_KEYS 64  // keys of a tile
#define PF_ROW (2 * PF_D)  // bytes

namespace {

// where the 16-byte piece p of a row lies, without bank conflicts: keys are
// read rows 8g + r (+ 4) of g, r < 4 at one piece, values rows 8g + r of two
// lane groups g at two
__device__ __forceinline__ int pf_key_piece(int row, int p) {
    return p ^ ((row & 3) | (row >> 3 & 3) << 2);
}
__device__ __forceinline__ int pf_value_piece(int row, int p) {
    return (((p >> 1) ^ ((row & 3) | (row >> 3 & 1) << 2)) << 1) | (p & 1);
}

// The sum of 64 weights of one column, of which a lane has those of keys
// 32c + 8*grp + 4h + r at [c][4h + r]: first the four of the keys that are equal
// in their last 4 bits, in order, then these by halves (8 apart, 4, 2, 1). A swap
// leaves one half's two operands in each half of the lanes.
__device__ __forceinline__ float add_in_halves(uint32_t a, uint32_t b) {
    return __uint_as_float(a) + __uint_as_float(b);
}
__device__ __forceinline__ float pf_key_sum(const float (&e)[2][8]) {
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const auto a = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(e[0][r]), __float_as_uint(e[0][4 + r]), false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(e[1][r]), __float_as_uint(e[1][4 + r]), false, false);
        v[r] = add_in_halves(a[0], a[1]) + __uint_as_float(b[0]) + __uint_as_float(b[1]);
    }
    float w[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const auto a = __builtin_amdgcn_permlane16_swap(
            __float_as_uint(v[r]), __float_as_uint(v[r + 2]), false, false);
        w[r] = add_in_halves(a[0], a[1]);
    }
    auto c = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(w[0]), __float_as_uint(w[1]), false, false);
    uint32_t x = __float_as_uint(add_in_halves(c[0], c[1]));
    c = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = __float_as_uint(add_in_halves(c[0], c[1]));
    c = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return add_in_halves(c[0], c[1]);
}

// 16 e4m3 bytes times their row's scale as 16 bf16
__device__ __forceinline__ void dequantize16(const uint4& b, float scale, uint4* out) {
    const uint32_t w[4] = {b.x, b.y, b.z, b.w};
    uint32_t* o = reinterpret_cast<uint32_t*>(out);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float f0, f1, f2, f3;
        fp8x4_to_f32(w[i], f0, f1, f2, f3);
        o[2 * i] = cvt_pk_bf16(f0 * scale, f1 * scale);
        o[2 * i + 1] = cvt_pk_bf16(f2 * scale, f3 * scale);
    }
}

}  // namespace

// HG: heads of a workgroup (four waves each); FP8C: pages are e4m3 with a scale
// a row.
template <int HG, bool FP8C>
__launch_bounds__(HG * 4 * WAVE_SIZE, 2)
__global__ void attention_prefill_kernel(
    bf16* __restrict__ out,             // [T, Hq, D]
    const bf16* __restrict__ q,         // [T, Hq, D] (rows strided)
    const bf16* __restrict__ k,         // [T, Hkv, D]
    const bf16* __restrict__ v,         // [T, Hkv, D]
    const int* __restrict__ cu_seqlens, // [B+1]
    const int* __restrict__ tile_seq,   // [ntiles] sequence of each tile
    const int* __restrict__ tile_off,   // [ntiles] its first row in the sequence
    float scale,
    int G, int Hkv, int head_groups, int64_t q_stride, int64_t k_stride, int64_t v_stride,
    const char* __restrict__ k_cache,   // [NB, Hkv, BS, D] or null
    const char* __restrict__ v_cache,
    const float* __restrict__ k_scale,  // [NB, Hkv, BS] (FP8C)
    const float* __restrict__ v_scale,
    const int* __restrict__ block_tables,  // [B, max_blocks] or null
    const int* __restrict__ cached_lens,   // [B] or null
    int block_size, int max_blocks) {
    constexpr int KT = PF_KEYS, NW = 4 * HG;
    constexpr int TILE = KT * PF_ROW;          // bytes of a key or value tile
    constexpr int MOVES = KT / 4;              // 1 KB transfers of one
    constexpr int MINE = (MOVES + NW - 1) / NW;
    const int per_tile = Hkv * head_groups;  // workgroups of a tile
    const int tile = gridDim.x / per_tile - 1 - blockIdx.x / per_tile;
    const int kvh = blockIdx.x % per_tile % Hkv, group = blockIdx.x % per_tile / Hkv;
    const int seq = tile_seq[tile], tile0 = tile_off[tile];
    const int seq_start = cu_seqlens[seq];
    const int seq_len = cu_seqlens[seq + 1] - seq_start;
    const int cached = cached_lens != nullptr ? cached_lens[seq] : 0;
    if (tile0 >= seq_len) return;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int head_in = group * HG + (wave >> 2); // of the kv head's G
    const bool has_head = head_in < G;
    const int row0 = tile0 + (wave & 3) * 16;      // of this wave
    const int Hq = G * Hkv, head = kvh * G + min(head_in, G - 1);

    __shared__ __attribute__((aligned(16))) char lds[2][2][TILE];

    bf16x8 qf[4];
    {
        const int r = min(row0 + col, seq_len - 1);
        const bf16* p = q + (int64_t)(seq_start + r) * q_stride + (int64_t)head * PF_D + grp * 8;
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const bf16x8*>(p + c * 32);
    }

    const int limit = min(seq_len, tile0 + QTILE);  // keys that the tile sees
    const int n_cached = (cached + KT - 1) / KT;
    const int n_tiles = n_cached + (limit + KT - 1) / KT;
    const int* table = block_tables != nullptr ? block_tables + (int64_t)seq * max_blocks : nullptr;

    // rows of a tile: transfer i has rows 4i..4i+3 of keys and of values, a lane 16
    // bytes of one; of bytes, it has 8 rows of keys, from KT / 8 on of values
    constexpr int PAGE_ROWS = FP8C ? (KT / 4 + NW - 1) / NW : MINE;
    auto page_row = [&](int j) {  // row in the tile whose page this lane looks up
        return FP8C ? (wave + j * NW) % (KT / 8) * 8 + (lane >> 3) : (wave + j * NW) * 4 + grp;
    };
    int pages[PAGE_ROWS];
    auto look_up = [&](int t) {
#pragma unroll
        for (int j = 0; j < PAGE_ROWS; ++j)
            if (t < n_cached)
                pages[j] = table[min(t * KT + page_row(j), cached - 1) / block_size];
    };
    uint4 bytes[FP8C ? PAGE_ROWS : 1];
    float scales[FP8C ? PAGE_ROWS : 1];

    auto issue = [&](int t) {
        const uint32_t at = lds_address(&lds[t & 1][0][0]);
        if (t < n_cached) {
#pragma unroll
            for (int j = 0; j < PAGE_ROWS; ++j) {
                const int i = wave + j * NW;
                if (i >= (FP8C ? KT / 4 : MOVES)) continue;
                const int r = page_row(j);
                const int pos = min(t * KT + r, cached - 1);
                const int64_t row =
                    ((int64_t)pages[j] * Hkv + kvh) * block_size + pos % block_size;
                if constexpr (FP8C) {
                    const bool of_keys = i < KT / 8;
                    bytes[j] = *reinterpret_cast<const uint4*>(
                        (of_keys ? k_cache : v_cache) + row * PF_D + (lane & 7) * 16);
                    scales[j] = (of_keys ? k_scale : v_scale)[row];
                } else {
                    const uint32_t to = __builtin_amdgcn_readfirstlane(at + i * 1024);
                    dma16((const bf16*)(k_cache + row * PF_ROW + pf_key_piece(r, col) * 16), to);
                    dma16((const bf16*)(v_cache + row * PF_ROW + pf_value_piece(r, col) * 16), to + TILE);
                }
            }
        } else {
            const int key0 = (t - n_cached) * KT;
#pragma unroll
            for (int j = 0; j < MINE; ++j) {
                if (wave + j * NW >= MOVES) continue;
                const int r = (wave + j * NW) * 4 + grp;
                const int64_t token = seq_start + min(key0 + r, limit - 1);
                const uint32_t to = __builtin_amdgcn_readfirstlane(at + (wave + j * NW) * 1024);
                dma16(k + token * k_stride + kvh * PF_D + pf_key_piece(r, col) * 8, to);
                dma16(v + token * v_stride + kvh * PF_D + pf_value_piece(r, col) * 8, to + TILE);
            }
        }
    };
    // tile t lies in LDS as far as this wave brings it; behind the last key lies
    // its row again: zero as values, as 0 times an infinity is none of their sum
    auto land = [&](int t) {
        const int rows = t < n_cached ? cached - t * KT : limit - (t - n_cached) * KT;
        if (rows < KT && !(FP8C && t < n_cached)) {
            wait_transfers<0>();
#pragma unroll
            for (int j = 0; j < MINE; ++j) {
                const int i = wave + j * NW, r = i * 4 + grp;
                if (i < MOVES && r >= rows)
                    *reinterpret_cast<uint4*>(&lds[t & 1][1][i * 1024 + lane * 16]) =
                        make_uint4(0, 0, 0, 0);
            }
        }
        if (FP8C && t < n_cached) {
#pragma unroll
            for (int j = 0; j < PAGE_ROWS; ++j) {
                const int i = wave + j * NW, r = page_row(j);
                if (i >= KT / 4) continue;
                const bool of_keys = i < KT / 8;
                uint4 x[2];
                dequantize16(bytes[j], scales[j], x);
                if (!of_keys && r >= rows) x[0] = x[1] = make_uint4(0, 0, 0, 0);
                char* at = lds[t & 1][of_keys ? 0 : 1] + r * PF_ROW;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int piece = (lane & 7) * 2 + h;
                    *reinterpret_cast<uint4*>(
                        at + (of_keys ? pf_key_piece(r, piece) : pf_value_piece(r, piece)) * 16) = x[h];
                }
            }
        }
    };

    float m = -INFINITY, l = 0.f;
    f32x4 acc[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[d] = (f32x4){0.f, 0.f, 0.f, 0.f};

    look_up(0);
    issue(0);
    look_up(1);
    // the queries' loads end here, not at their first use inside the loop
#pragma unroll
    for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[c]));

    // fragment addresses: row i of a product's first operand is key 8(i/4) + i%4
    // of 32 (+ 4 in the second), piece 4c + grp, so that a lane's scores are those
    // of keys 8*grp..8*grp+7; values of these rows, columns 16d + (col%4)*4
    const int k_row = (col >> 2) * 8 + (col & 3);
    int key_at[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        key_at[c] = k_row * PF_ROW + pf_key_piece(k_row, c * 4 + grp) * 16;
    const int v_row = grp * 8 + (col >> 2);
    const int value_at = v_row * PF_ROW + ((col >> 1) & 1) * 16 + (col & 1) * 8;

    for (int t = 0; t < n_tiles; ++t) {
        land(t);
        dma_barrier();
        if (t + 1 < n_tiles) {
            issue(t + 1);
            look_up(t + 2);
        }
        const bool fresh = t >= n_cached;
        const int key0 = (fresh ? t - n_cached : t) * KT;
        // rows of this wave behind all keys of the tile: nothing to do
        if (!has_head || (fresh && key0 > row0 + 15) || row0 >= seq_len) continue;
        const char* keys = lds[t & 1][0];
        const char* vals = lds[t & 1][1];

        float s[2][8];  // scores of keys 32c + 8*grp + j
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    p = mfma16(*reinterpret_cast<const bf16x8*>(
                                   keys + key_at[d] + (c * 32 + h * 4) * PF_ROW), qf[d], p);
#pragma unroll
                for (int r = 0; r < 4; ++r) s[c][h * 4 + r] = p[r] * scale;
            }

        // keys that some row of this wave does not see
        if (key0 + KT > (fresh ? row0 + 1 : cached)) {
            const int most = fresh ? row0 + col : cached - 1;
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (key0 + c * 32 + grp * 8 + j > most) s[c][j] = -INFINITY;
        }

        float top = s[0][0];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int j = 0; j < 8; ++j) top = fmaxf(top, s[c][j]);
        top = column_max(top);
        float factor = 1.f;
        if (__any(top > m)) {
            const float m_new = fmaxf(m, top);
            factor = __expf(m - (m_new == -INFINITY ? 0.f : m_new));
            m = m_new;
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[d][r] *= factor;
        }
        bf16x8 p[2];
        const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float* e = s[c];
#pragma unroll
            for (int j = 0; j < 8; ++j) e[j] = __expf(e[j] - base);
            p[c] = as_frag(make_uint4(cvt_pk_bf16(e[0], e[1]), cvt_pk_bf16(e[2], e[3]),
                                      cvt_pk_bf16(e[4], e[5]), cvt_pk_bf16(e[6], e[7])));
        }
        l = fmaf(l, factor, pf_key_sum(s));

#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const int at = value_at + ((d ^ ((v_row & 3) | (v_row >> 3 & 1) << 2)) << 5);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16* lo = reinterpret_cast<const bf16*>(vals + at + c * 32 * PF_ROW);
                acc[d] = mfma16(tr_pair(lo, lo + 4 * PF_D), p[c], acc[d]);
            }
        }
    }

    const int r = row0 + col;
    if (!has_head || r >= seq_len || l <= 0.f) return;
    const float inv = 1.f / l;
    bf16* o = out + ((int64_t)(seq_start + r) * Hq + head) * PF_D + grp * 4;
#pragma unroll
    for (int d = 0; d < 8; ++d)
        *reinterpret_cast<uint2*>(o + d * 16) =
            make_uint2(cvt_pk_bf16(acc[d][0] * inv, acc[d][1] * inv),
                       cvt_pk_bf16(acc[d][2] * inv, acc[d][3] * inv));
}

extern "C" hipError_t launch_attention_prefill(
    void* out, const void* q, const void* k, const void* v,
    const int* cu_seqlens, const int* tile_seq, const int* tile_off,
    int ntiles, float scale, int Hq, int Hkv, int D, int64_t q_stride,
    int64_t k_stride, int64_t v_stride, const void* k_cache,
    const void* v_cache, const float* k_scale, const float* v_scale,
    const int* block_tables, const int* cached_lens,
    int block_size, int max_blocks, hipStream_t stream) {
    if (D != PF_D) return hipErrorNotSupported;
    if (Hkv <= 0 || Hq % Hkv != 0) return hipErrorInvalidValue;
    if (ntiles <= 0) return hipSuccess;
    const int G = Hq / Hkv;
#define LAUNCH(HG)                                                           \
    do {                                                                       \
        const int groups = (G + HG - 1) / HG;                                  \
        const dim3 grid(Hkv * groups * ntiles), block(HG * 4 * WAVE_SIZE);           \
        if (k_scale != nullptr)                                                \
            attention_prefill_kernel<HG, true><<<grid, block, 0, stream>>>(\
                (bf16*)out, (const bf16*)q, (const bf16*)k, (const bf16*)v,    \
                cu_seqlens, tile_seq, tile_off, scale, G, Hkv, groups,     \
                q_stride, k_stride, v_stride, (const char*)k_cache,            \
                (const char*)v_cache, k_scale, v_scale, block_tables,          \
                cached_lens, block_size, max_blocks);                          \
        else                                                                   \
            attention_prefill_kernel<HG, false><<<grid, block, 0, stream>>>(\
                (bf16*)out, (const bf16*)q, (const bf16*)k, (const bf16*)v,    \
                cu_seqlens, tile_seq, tile_off, scale, G, Hkv, groups,     \
                q_stride, k_stride, v_stride, (const char*)k_cache,            \
                (const char*)v_cache, k_scale, v_scale, block_tables,          \
                cached_lens, block_size, max_blocks);                          \
    } while (0)
    // Heads of a workgroup: one where that many workgroups run at once or nearly
    // (512 do), two beyond; with cached rows, where keys are many for all rows, as
    // many as still give work to half of the 256 CUs. One head a kv head has two,
    // whose idle waves bring keys. us with 1 / 2 / 3 / 4 heads:
    //   32:8 heads   300 tokens 10 / 12 / 15 / 17, 1000 26 / 29 / 36 / 42, 1600 46 /
    //     50 / 60 / 67, 2000 70 / 64 / 83 / 83, 4096 227 / 189 / 275 / 189, 32 x
    //     66-128 27 / 23 / 33 / 26; after 2000: 3 x 150 73 / 66 / 77 / 85, 6 x 150 132
    //     / 100 / 153 / 90 (e4m3 170 / 153 / 172 / 99); 4000 after 4032 693 / 503 /
    //     789 / 464
    //   24:8 heads   4000 tokens 170 / 164 / 147 / 152
    //   28:4 heads   1500 tokens 38 / 46 / 55 / 61, 3000 119 / 112 / 118 / 116; 3000
    //     after 1000 in e4m3 233 / 231 / 203 / 179
    //   32:32 heads  2000 tokens 68 / 65 / 94 / 85
    auto groups_of = [&](int heads) { return ntiles * Hkv * ((G + heads - 1) / heads); };
    if (cached_lens != nullptr && G > 2 && groups_of(4) >= 128) {
        if (G == 3 || G == 5 || G == 6) LAUNCH(3);
        else LAUNCH(4);
    } else if (G > 1 && (cached_lens != nullptr ? groups_of(2) < 128 : groups_of(1) <= 800)) {
        LAUNCH(1);
    } else if (G == 3) {
        LAUNCH(3);
    } else {
        LAUNCH(2);
    }
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}
