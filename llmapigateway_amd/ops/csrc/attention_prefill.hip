// Causal prompt attention for gfx950 (MFMA bf16), varlen with GQA, over the
// step's own rows and, where a sequence has cached context (prefix caching,
// chunked prefill), over its pages in front of them.
//
// Produces the prompt phase (TTFT) the reference delegated upstream.
//
// - A workgroup has 64 query rows of up to four heads of one kv head: each wave
//   32 rows of one head, so that a key and value tile staged once serves 256
//   query columns, and a fragment read from LDS two products.
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
//   that moves only past 2^8 takes 163 us instead of 185 for 4096 tokens, but
//   rounds the largest weights, too: over 4000 keys the weights' share of the error
//   is 1.6e-3 then, 1.25e-3 so.)
// - Blocks of one kv head follow each other at the distance of the XCDs, and
//   late tiles, which see the most keys, start first.
//
// One layer, 32 query and 8 kv heads; before: 64 rows and one head a workgroup,
// keys and values through registers, weights through LDS:
//   4096 tokens                   1117 us -> 185 us (743 TFLOP/s)
//   4000 tokens after 4032        2371    -> 503    (786), e4m3 pages the same
//   9 x 117-213 tokens after 1984  428    -> 102
//   32 x 66-128 tokens              46    ->  24
//   37 tokens                      6.6    -> 6.3
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

// HG: heads of a workgroup (two waves each); FP8C: pages are e4m3 with a scale
// a row.
template <int HG, bool FP8C>
__launch_bounds__(HG * 2 * WAVE_SIZE, 2)
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
    constexpr int KT = PF_KEYS, NW = 2 * HG, NQ = 2;
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
    const int head_in = group * HG + (wave >> 1);  // of the kv head's G
    const bool has_head = head_in < G;
    const int row0 = tile0 + (wave & 1) * 32;      // of this wave
    const int Hq = G * Hkv, head = kvh * G + min(head_in, G - 1);

    __shared__ __attribute__((aligned(16))) char lds[2][2][TILE];

    bf16x8 qf[NQ][4];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int r = min(row0 + n * 16 + col, seq_len - 1);
        const bf16* p = q + (int64_t)(seq_start + r) * q_stride + (int64_t)head * PF_D + grp * 8;
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[n][c] = *reinterpret_cast<const bf16x8*>(p + c * 32);
    }

    const int limit = min(seq_len, tile0 + QTILE);  // keys that the tile sees
    const int n_cached = (cached + KT - 1) / KT;
    const int n_tiles = n_cached + (limit + KT - 1) / KT;
    const int* table = block_tables != nullptr ? block_tables + (int64_t)seq * max_blocks : nullptr;

    // rows of a tile: transfer i has rows 4i..4i+3, a lane 16 bytes of one; of
    // bytes, 8 lanes have a row and a wave 8 rows
    constexpr int PAGE_ROWS = FP8C ? (KT / 8 + NW - 1) / NW : MINE;
    auto page_row = [&](int j) {  // row in the tile whose page this lane looks up
        return FP8C ? (wave + j * NW) * 8 + (lane >> 3) : (wave + j * NW) * 4 + grp;
    };
    int pages[PAGE_ROWS];
    auto look_up = [&](int t) {
#pragma unroll
        for (int j = 0; j < PAGE_ROWS; ++j)
            if (t < n_cached)
                pages[j] = table[min(t * KT + page_row(j), cached - 1) / block_size];
    };
    uint4 kb[FP8C ? PAGE_ROWS : 1], vb[FP8C ? PAGE_ROWS : 1];
    float ks[FP8C ? PAGE_ROWS : 1], vs[FP8C ? PAGE_ROWS : 1];

    auto issue = [&](int t) {
        const uint32_t at = lds_address(&lds[t & 1][0][0]);
        if (t < n_cached) {
#pragma unroll
            for (int j = 0; j < PAGE_ROWS; ++j) {
                const int r = page_row(j);
                if (r - (FP8C ? lane >> 3 : grp) >= KT) continue;  // uniform
                const int pos = min(t * KT + r, cached - 1);
                const int64_t row =
                    ((int64_t)pages[j] * Hkv + kvh) * block_size + pos % block_size;
                if constexpr (FP8C) {
                    kb[j] = *reinterpret_cast<const uint4*>(k_cache + row * PF_D + (lane & 7) * 16);
                    vb[j] = *reinterpret_cast<const uint4*>(v_cache + row * PF_D + (lane & 7) * 16);
                    ks[j] = k_scale[row];
                    vs[j] = v_scale[row];
                } else {
                    const uint32_t to = __builtin_amdgcn_readfirstlane(at + (wave + j * NW) * 1024);
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
    // tile t lies in LDS as far as this wave brings it
    auto land = [&](int t) {
        if (FP8C && t < n_cached) {
            char* at = &lds[t & 1][0][0];
#pragma unroll
            for (int j = 0; j < PAGE_ROWS; ++j) {
                const int r = page_row(j);
                if (r - (lane >> 3) >= KT) continue;
                uint4 x[2];
                dequantize16(kb[j], ks[j], x);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<uint4*>(
                        at + r * PF_ROW + pf_key_piece(r, (lane & 7) * 2 + h) * 16) = x[h];
                dequantize16(vb[j], vs[j], x);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<uint4*>(
                        at + TILE + r * PF_ROW + pf_value_piece(r, (lane & 7) * 2 + h) * 16) = x[h];
            }
        }
    };

    float m[NQ], l[NQ];
    f32x4 acc[NQ][8];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m[n] = -INFINITY;
        l[n] = 0.f;
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[n][d] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    look_up(0);
    issue(0);
    look_up(1);
    // the queries' loads end here, not at their first use inside the loop
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
        for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[n][c]));

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
        // behind the last key lies its row again: 0 times an infinity is none of
        // the values' sum
        const int rows = (fresh ? limit : cached) - key0;
        if (rows < KT) {
            for (int i = rows * (PF_ROW / 16) + threadIdx.x; i < TILE / 16; i += NW * WAVE_SIZE)
                reinterpret_cast<uint4*>(lds[t & 1][1])[i] = make_uint4(0, 0, 0, 0);
            lds_barrier();
        }
        // rows of this wave behind all keys of the tile: nothing to do
        if (!has_head || (fresh && key0 > row0 + 31) || row0 >= seq_len) continue;
        const char* keys = lds[t & 1][0];
        const char* vals = lds[t & 1][1];

        float s[NQ][2][8];  // scores of keys 32c + 8*grp + j
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 p[NQ];
#pragma unroll
                for (int n = 0; n < NQ; ++n) p[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const bf16x8 kf =
                        *reinterpret_cast<const bf16x8*>(keys + key_at[d] + (c * 32 + h * 4) * PF_ROW);
#pragma unroll
                    for (int n = 0; n < NQ; ++n) p[n] = mfma16(kf, qf[n][d], p[n]);
                }
#pragma unroll
                for (int n = 0; n < NQ; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[n][c][h * 4 + r] = p[n][r] * scale;
            }

        // keys that some row of this wave does not see
        const int seen = fresh ? row0 + 1 : cached;
        if (key0 + KT > seen) {
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                const int most = fresh ? row0 + n * 16 + col : cached - 1;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (key0 + c * 32 + grp * 8 + j > most) s[n][c][j] = -INFINITY;
            }
        }

        float top[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            float x = s[n][0][0];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < 8; ++j) x = fmaxf(x, s[n][c][j]);
            top[n] = column_max(x);
        }
        float factor[NQ] = {1.f, 1.f};
        if (__any(top[0] > m[0] || top[1] > m[1])) {
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                const float m_new = fmaxf(m[n], top[n]);
                factor[n] = __expf(m[n] - (m_new == -INFINITY ? 0.f : m_new));
                m[n] = m_new;
#pragma unroll
                for (int d = 0; d < 8; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[n][d][r] *= factor[n];
            }
        }
        bf16x8 p[NQ][2];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            const float base = m[n] == -INFINITY ? 0.f : m[n];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float* e = s[n][c];
#pragma unroll
                for (int j = 0; j < 8; ++j) e[j] = __expf(e[j] - base);
                p[n][c] = as_frag(make_uint4(
                    cvt_pk_bf16(e[0], e[1]), cvt_pk_bf16(e[2], e[3]),
                    cvt_pk_bf16(e[4], e[5]), cvt_pk_bf16(e[6], e[7])));
            }
            l[n] = fmaf(l[n], factor[n], pf_key_sum(s[n]));
        }

#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const int at = value_at + ((d ^ ((v_row & 3) | (v_row >> 3 & 1) << 2)) << 5);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16* lo = reinterpret_cast<const bf16*>(vals + at + c * 32 * PF_ROW);
                const bf16x8 vf = tr_pair(lo, lo + 4 * PF_D);
#pragma unroll
                for (int n = 0; n < NQ; ++n) acc[n][d] = mfma16(vf, p[n][c], acc[n][d]);
            }
        }
    }

    if (!has_head) return;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int r = row0 + n * 16 + col;
        if (r >= seq_len || l[n] <= 0.f) continue;
        const float inv = 1.f / l[n];
        bf16* o = out + ((int64_t)(seq_start + r) * Hq + head) * PF_D + grp * 4;
#pragma unroll
        for (int d = 0; d < 8; ++d)
            *reinterpret_cast<uint2*>(o + d * 16) =
                make_uint2(cvt_pk_bf16(acc[n][d][0] * inv, acc[n][d][1] * inv),
                           cvt_pk_bf16(acc[n][d][2] * inv, acc[n][d][3] * inv));
    }
}

extern "C" hipError_t launch_attention_prefill(
    void* out, const void* q, const void* k, const void* v,
    const int* cu_seqlens, const int* tile_seq, const int* tile_off,
    int ntiles, int nseq, float scale, int Hq, int Hkv, int D, int64_t q_stride,
    int64_t k_stride, int64_t v_stride, const void* k_cache,
    const void* v_cache, const float* k_scale, const float* v_scale,
    const int* block_tables, const int* cached_lens,
    int block_size, int max_blocks, hipStream_t stream) {
    if (D != PF_D) return hipErrorNotSupported;
    if (Hkv <= 0 || Hq % Hkv != 0) return hipErrorInvalidValue;
    if (ntiles <= 0) return hipSuccess;
    const int G = Hq / Hkv;
#define LAUNCH(HG)                                                       \
    do {                                                                       \
        const int groups = (G + HG - 1) / HG;                                  \
        const dim3 grid(Hkv * groups * ntiles), block(HG * 2 * WAVE_SIZE);      \
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
    // Heads of a workgroup, by how many workgroups of four heads there would be.
    // Four (three where that divides the group better) where they fill the 256
    // CUs; two where CUs would idle, or where sequences are short and latency
    // counts. 32:8 heads, us with 4 / 2 / 1 heads: 4096 tokens 189 / 199 / 329, 9 x
    // 117-213 after 1984 106 / 110 / 231, 1000 tokens 44 / 34 / 44, 32 x 66-128 27 /
    // 24 / 35, 300 tokens 18 / 13 / 16, 37 tokens 7.9 / 6.6 / 7.2. One head a kv
    // head: the waves without one bring keys (32 heads, 2000 tokens 89 us with two,
    // 93 with one; 150 tokens after 1000 46 and 66).
    const int full = ntiles * Hkv * ((G + 3) / 4);
    const bool short_keys = cached_lens == nullptr && ntiles <= 4 * nseq;
    if (G <= 2 || full < 160 || short_keys) LAUNCH(2);
    else if (G == 3 || G == 5 || G == 6) LAUNCH(3);
    else LAUNCH(4);
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}
