// Paged decode attention for gfx950 (GQA, bf16 or e4m3 KV cache).
//
// Replaces the per-token generation the reference gateway delegated to its
// remote providers. Memory-bound: the whole KV history of each sequence is
// read once per step, so everything here serves the stream.
//
// - A workgroup has a span of one sequence's context for one kv head; its
//   four waves take that span's tiles (16 keys in bf16, 32 in e4m3: 4 KB of
//   keys and 4 KB of values) in turn, each for itself: a ring of two tiles a
//   wave in LDS, filled by transfers that need no registers, waited for by
//   count, no barrier until the waves' shares meet at the end. 64 KB of LDS a
//   workgroup let two workgroups share a CU, with 64 KB in flight there.
// - All G = Hq/Hkv query heads of the kv head are the columns of one product
//   S^T = K Q^T (zero columns up to 16), so a lane's softmax state is one
//   scalar, and the weights as they stand are the operand of O^T = V^T P^T,
//   whose V fragments come from LDS by transposing reads. Weights stay fp32:
//   they enter as the sum of two bf16 (relative error 2^-17). An e4m3 value
//   is a bf16 value, so pages of bytes lose nothing either; their scales
//   multiply scores and weights in fp32.
// - Contexts are split where sequences and heads alone leave CUs idle. The
//   number of splits is fixed by shapes (a captured graph must hold for any
//   context), the span is cut on the device from the context's length, and
//   spans without keys end at once; a second kernel adds the partials up.
//
// One layer's attention with 32 query and 8 kv heads, contexts ragged from half
// of the stated one up; "was": one key a lane, FMA, spans of 2048; "floor": the
// pages' bytes at the 6.1 TB/s that the best reading kernel here reaches.
//     1 x  611          floor  0.4 us   was  65   now  6.9 (two launches)
//     3 x 7801          floor 11.8      was 166   now 19.1
//    11 x 1500          floor  8.3      was 125   now 18
//    45 x  900 (28:4)   floor 10.2      was 102   now 15.9
//   256 x  192          floor 24.7      was  49   now 30.2
//   120 x 2000, e4m3    floor 62        was 220   now 70.8
// What is left: the ramp (page, transfer, one tile's chain, about 4 us) and the
// second kernel (3 us) where little is read; the rate of the reads where much is.

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

#define DECODE_D 128
#define MAX_G 8
// four waves: with two a span of 900 keys takes 22.9 us instead of 16.7, with
// eight 256 contexts of 192 take 44 us instead of 33; a third tile in the ring
// gains nothing
#define DECODE_WAVES 4
#define MIN_SPAN 64  // keys of a workgroup's round (4 waves x 16)

namespace {

typedef int i32x2 __attribute__((ext_vector_type(2)));

// A wave's tile: keys, then values, rows of 128 elements. Rows lie in LDS as
// they come (lane l's 16 bytes at 16 * l of each 1 KB transfer), the 16-byte
// pieces of a row in an order that keeps the reads free of bank conflicts:
// keys by pieces (16 rows at one piece), values by column blocks of 16.
template <bool FP8>
struct DecodeTile {
    static constexpr int KEYS = FP8 ? 32 : 16;
    static constexpr int SUBS = KEYS / 16;
    static constexpr int ROW = FP8 ? DECODE_D : 2 * DECODE_D;  // bytes
    static constexpr int PIECES = ROW / 16;                    // of 16 bytes
    static constexpr int BYTES = KEYS * ROW;                   // 4 KB
    static constexpr int ROWS_A_TRANSFER = 1024 / ROW;
    static constexpr int TRANSFERS = BYTES / 1024;             // of keys, and of values
    static constexpr int SLOT = 2 * BYTES + (FP8 ? 256 : 0);   // scales behind
    static constexpr int IN_FLIGHT = 2 * TRANSFERS + (FP8 ? 1 : 0);

    // where piece p of a row lies
    static __device__ __forceinline__ int key_piece(int row, int p) {
        return FP8 ? p ^ ((row >> 1) & 7) : p ^ (row & 15);
    }
    static __device__ __forceinline__ int value_piece(int row, int p) {
        return FP8 ? p ^ ((row >> 1) & 7) : (((p >> 1) ^ (row & 7)) << 1) | (p & 1);
    }
};

// keys of one split of a context of length L
__device__ __forceinline__ int span_of(int L, int nsplit) {
    const int even = (L + nsplit - 1) / nsplit;
    return (even + MIN_SPAN - 1) / MIN_SPAN * MIN_SPAN;
}

// 8 e4m3 bytes as 8 bf16 (exact)
__device__ __forceinline__ bf16x8 e4m3_frag(uint32_t lo, uint32_t hi) {
    typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
    uint4 v;
    b16x2* p = reinterpret_cast<b16x2*>(&v);
    p[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false);
    p[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true);
    p[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false);
    p[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true);
    return as_frag(v);
}

__device__ __forceinline__ f32x4 mfma16_k16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

}  // namespace

// PAGED: pages hold whole tiles (block_size a multiple of the tile), so a tile
// has one page; else every row looks its page up. SPLIT: partials instead of
// the output.
template <bool FP8, bool SPLIT, bool PAGED>
__launch_bounds__(DECODE_WAVES* WAVE_SIZE)
__global__ void attention_decode_kernel(
    bf16* __restrict__ out,                // [B, Hq, D]
    const bf16* __restrict__ q,            // [B, Hq, D], rows q_stride apart
    const char* __restrict__ k_cache,      // [NB, Hkv, BS, D] bf16 | e4m3
    const char* __restrict__ v_cache,
    const float* __restrict__ k_scale,     // [NB, Hkv, BS] (FP8)
    const float* __restrict__ v_scale,
    const int* __restrict__ block_tables,  // [B, max_blocks]
    const int* __restrict__ context_lens,  // [B]
    float scale_log2,                      // scale * log2(e)
    int Hkv, int G, int block_size, int max_blocks, int64_t q_stride,
    float* __restrict__ part_acc,          // [B, Hq, nsplit, D] (SPLIT)
    float* __restrict__ part_ml,           // [B, Hq, nsplit, 2] (SPLIT)
    int nsplit) {
    using Tile = DecodeTile<FP8>;
    constexpr int W = DECODE_WAVES, NB = 2;  // waves, and tiles of each in LDS
    const int seq = blockIdx.x, kvh = blockIdx.y, split = SPLIT ? blockIdx.z : 0;
    const int L = context_lens[seq];
    const int span = SPLIT ? span_of(L, nsplit) : L;
    const int start = split * span, stop = min(L, start + span);
    if (start >= stop) return;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int* table = block_tables + (size_t)seq * max_blocks;

    __shared__ __attribute__((aligned(16))) char ring[W][NB][Tile::SLOT];
    const uint32_t ring_at = __builtin_amdgcn_readfirstlane(lds_address(&ring[wave][0][0]));

    const int tiles = (stop - start + Tile::KEYS - 1) / Tile::KEYS;
    const int mine = wave < tiles ? (tiles - wave + W - 1) / W : 0;

    // Pages are read once, past the caches (120 contexts of 2000 in e4m3 70.8 us, 80
    // without; 256 of 192 30.2 and 33.7; 256 of 1500 195 and 217), unless the
    // context begins with the page of the one before or behind it: then the caches
    // have a common part for both (24 contexts on the same pages take 21 us so, 31
    // past the caches). What that look misses costs time only.
    const int before = seq > 0 ? -max_blocks : 0;
    const int behind = seq + 1 < (int)gridDim.x ? max_blocks : 0;
    const int first = table[0];
    const bool once = (before == 0 || table[before] != first) &
                      (behind == 0 || table[behind] != first);

    // transfer of tile i of this wave; page: of its first key (PAGED)
    const int t_row = lane / Tile::PIECES, t_piece = lane % Tile::PIECES;
    auto first_key = [&](int i) { return start + (wave + i * W) * Tile::KEYS; };
    auto page_of = [&](int i) { return PAGED ? table[first_key(i) / block_size] : 0; };
    auto fetch = [&](int i, int page) {
        const int key0 = first_key(i);
        const uint32_t at = ring_at + (i % NB) * Tile::SLOT;
        const int64_t page_row = ((int64_t)page * Hkv + kvh) * block_size;
        const int off0 = PAGED ? key0 % block_size : 0;
        const int most = stop - 1 - key0;  // the last row that is a key
        // waves read a slot's last values before it is filled again
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        auto row_of = [&](int r) -> int64_t {
            r = min(r, most);
            if (PAGED) return page_row + off0 + r;
            const int pos = key0 + r;
            return ((int64_t)table[pos / block_size] * Hkv + kvh) * block_size + pos % block_size;
        };
        int64_t rows[Tile::TRANSFERS];
#pragma unroll
        for (int j = 0; j < Tile::TRANSFERS; ++j)
            rows[j] = row_of(j * Tile::ROWS_A_TRANSFER + t_row);
        int64_t scale_row = 0;
        if (FP8) scale_row = row_of(lane & 31);
        auto key = [&](int j) {
            const int r = j * Tile::ROWS_A_TRANSFER + t_row;
            return reinterpret_cast<const bf16*>(
                k_cache + rows[j] * Tile::ROW + Tile::key_piece(r, t_piece) * 16);
        };
        auto value = [&](int j) {
            const int r = j * Tile::ROWS_A_TRANSFER + t_row;
            return reinterpret_cast<const bf16*>(
                v_cache + rows[j] * Tile::ROW + Tile::value_piece(r, t_piece) * 16);
        };
        if (once) {
#pragma unroll
            for (int j = 0; j < Tile::TRANSFERS; ++j) dma16_once(key(j), at + j * 1024);
#pragma unroll
            for (int j = 0; j < Tile::TRANSFERS; ++j)
                dma16_once(value(j), at + Tile::BYTES + j * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < Tile::TRANSFERS; ++j) dma16(key(j), at + j * 1024);
#pragma unroll
            for (int j = 0; j < Tile::TRANSFERS; ++j)
                dma16(value(j), at + Tile::BYTES + j * 1024);
        }
        if (FP8) dma4((lane < 32 ? k_scale : v_scale) + scale_row, at + 2 * Tile::BYTES);
    };

    int page = 0;
    if (mine > 0) page = page_of(0);

    // queries, the second operand of S^T: lane's 8 dims of its head. In bf16
    // step c covers dims 32c..32c+31; from bytes, two steps share a group's 16
    // bytes, so steps 2p and 2p+1 cover its dims (4p + group) * 16 + 0..7 and
    // 8..15.
    bf16x8 qf[4];
    {
        const bf16* qrow = q + (int64_t)seq * q_stride + (int64_t)(kvh * G + col) * DECODE_D;
        const bool wide = (((uintptr_t)q | (uint64_t)(q_stride * 2)) & 15) == 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int d = FP8 ? ((c >> 1) * 4 + grp) * 16 + (c & 1) * 8 : c * 32 + grp * 8;
            uint4 v = {0, 0, 0, 0};
            if (col < G) {
                if (wide) {
                    v = *reinterpret_cast<const uint4*>(qrow + d);
                } else {
                    const uint16_t* s = reinterpret_cast<const uint16_t*>(qrow + d);
                    uint32_t* o = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        o[j] = (uint32_t)s[2 * j] | ((uint32_t)s[2 * j + 1] << 16);
                }
            }
            qf[c] = as_frag(v);
        }
    }

    float m = -INFINITY, l = 0.f;
    f32x4 acc[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[d] = (f32x4){0.f, 0.f, 0.f, 0.f};

    int fetched = 0;
#pragma unroll
    for (int i = 0; i < NB - 1; ++i)
        if (i < mine) {
            fetch(i, page);
            ++fetched;
            if (fetched < mine) page = page_of(fetched);
        }
    // the queries' loads end here: a wait for them inside the loop would be a
    // wait for every transfer
#pragma unroll
    for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(qf[c]));
    for (int i = 0; i < mine; ++i) {
        if (fetched < mine) {
            fetch(fetched, page);
            ++fetched;
            if (fetched < mine) page = page_of(fetched);
        }
        const int ahead = fetched - 1 - i;
        if (ahead >= 1) wait_transfers<Tile::IN_FLIGHT>();
        else wait_transfers<0>();

        const char* keys = ring[wave][i % NB];
        const char* vals = keys + Tile::BYTES;
        const int key0 = first_key(i);

        // S^T: rows are keys, columns heads
        f32x4 s[Tile::SUBS];
#pragma unroll
        for (int u = 0; u < Tile::SUBS; ++u) {
            s[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
            const int row = u * 16 + col;
            if (FP8) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const uint4 b = *reinterpret_cast<const uint4*>(
                        keys + row * Tile::ROW + Tile::key_piece(row, p * 4 + grp) * 16);
                    s[u] = mfma16(e4m3_frag(b.x, b.y), qf[2 * p], s[u]);
                    s[u] = mfma16(e4m3_frag(b.z, b.w), qf[2 * p + 1], s[u]);
                }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint4 b = *reinterpret_cast<const uint4*>(
                        keys + row * Tile::ROW + Tile::key_piece(row, c * 4 + grp) * 16);
                    s[u] = mfma16(as_frag(b), qf[c], s[u]);
                }
            }
        }

        float p[4 * Tile::SUBS];
        float top = -INFINITY;
#pragma unroll
        for (int u = 0; u < Tile::SUBS; ++u) {
            float4 ks = {1.f, 1.f, 1.f, 1.f};
            if (FP8) ks = *reinterpret_cast<const float4*>(vals + Tile::BYTES + (u * 16 + grp * 4) * 4);
            const float* ksf = reinterpret_cast<const float*>(&ks);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = s[u][r] * scale_log2;
                if (FP8) v *= ksf[r];
                if (key0 + u * 16 + grp * 4 + r >= stop) v = -INFINITY;
                p[u * 4 + r] = v;
                top = fmaxf(top, v);
            }
        }
        const float m_new = fmaxf(m, column_max(top));
        const float base = m_new == -INFINITY ? 0.f : m_new;
        const float factor = __builtin_amdgcn_exp2f(m - base);
        m = m_new;
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 4 * Tile::SUBS; ++r) {
            p[r] = __builtin_amdgcn_exp2f(p[r] - base);
            sum += p[r];
        }
        l = l * factor + sum;  // of this lane's keys
#pragma unroll
        for (int d = 0; d < 8; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[d][r] *= factor;

        if constexpr (FP8) {
            const float* vs = reinterpret_cast<const float*>(vals + Tile::BYTES + 128);
#pragma unroll
            for (int u = 0; u < Tile::SUBS; ++u) {
                const float4 sc = *reinterpret_cast<const float4*>(vs + u * 16 + grp * 4);
                p[u * 4] *= sc.x;
                p[u * 4 + 1] *= sc.y;
                p[u * 4 + 2] *= sc.z;
                p[u * 4 + 3] *= sc.w;
            }
            bf16x8 hi, lo;
            split_frag(p, hi, lo);
            // keys of a lane group: 4g..4g+3 and 16+4g..16+4g+3, as p has them
            const int i8 = col >> 1;
            const int row = i8 < 4 ? grp * 4 + i8 : 12 + grp * 4 + i8;
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const char* at = vals + row * Tile::ROW + Tile::value_piece(row, d) * 16 + (col & 1) * 8;
                const i32x2 b = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                    (__attribute__((address_space(3))) i32x2*)at);
                const bf16x8 v = e4m3_frag(b[0], b[1]);
                acc[d] = mfma16(v, hi, acc[d]);
                acc[d] = mfma16(v, lo, acc[d]);
            }
        } else {
            union { uint32_t u[2]; bf16x4 v; } hi, lo;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                hi.u[j] = cvt_pk_bf16(p[2 * j], p[2 * j + 1]);
                float a, b;
                unpack2(hi.u[j], a, b);
                lo.u[j] = cvt_pk_bf16(p[2 * j] - a, p[2 * j + 1] - b);
            }
            const int row = grp * 4 + (col >> 2);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const char* at = vals + row * Tile::ROW +
                                 Tile::value_piece(row, d * 2 + ((col >> 1) & 1)) * 16 + (col & 1) * 8;
                const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) bf16x4*)at);
                acc[d] = mfma16_k16(v, hi.v, acc[d]);
                acc[d] = mfma16_k16(v, lo.v, acc[d]);
            }
        }
    }
    l = column_sum(l);

    // ---- the waves' shares meet (a wave without tiles has m = -inf) ----
    // acc[d][r] is dim 16d + 4*grp + r of head col
    __syncthreads();  // all tiles read
    float* share = reinterpret_cast<float*>(&ring[0][0][0]);  // [W][G][2 + D]
    constexpr int SHARE = 4 + DECODE_D;  // rows of 16-byte multiples
    if (col < G) {
        float* mine_at = share + ((size_t)wave * G + col) * SHARE;
        if (grp == 0) {
            mine_at[0] = m;
            mine_at[1] = l;
        }
#pragma unroll
        for (int d = 0; d < 8; ++d)
            *reinterpret_cast<f32x4*>(mine_at + 4 + d * 16 + grp * 4) = acc[d];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < G * (DECODE_D / 4); i += W * WAVE_SIZE) {
        const int g = i / (DECODE_D / 4), d = (i % (DECODE_D / 4)) * 4;
        float gm = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) gm = fmaxf(gm, share[(w * G + g) * SHARE]);
        const float base = gm == -INFINITY ? 0.f : gm;
        float gl = 0.f;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float* at = share + (w * G + g) * SHARE;
            const float f = __builtin_amdgcn_exp2f(at[0] - base);
            gl += f * at[1];
            const f32x4 a = *reinterpret_cast<const f32x4*>(at + 4 + d);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] += f * a[r];
        }
        // 0 times an infinity, as the low half of a weight or that of a row behind
        // the last key, is not what the sum of weights and values has there
        if (!FP8 && gl == gl && !(o[0] - o[0] + o[1] - o[1] + o[2] - o[2] + o[3] - o[3] == 0.f)) {
            float odd[4] = {0.f, 0.f, 0.f, 0.f};
            for (int key = start; key < stop; ++key) {
                const int64_t at = ((int64_t)table[key / block_size] * Hkv + kvh) * block_size +
                                   key % block_size;
                const uint2 raw = *reinterpret_cast<const uint2*>(v_cache + at * Tile::ROW + d * 2);
                float v[4];
                unpack2(raw.x, v[0], v[1]);
                unpack2(raw.y, v[2], v[3]);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (v[r] - v[r] != 0.f) odd[r] += v[r];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (odd[r] != 0.f) o[r] = odd[r];
        }
        const size_t row = (size_t)seq * Hkv * G + kvh * G + g;
        if (SPLIT) {
            const size_t pb = row * nsplit + split;
            *reinterpret_cast<f32x4*>(part_acc + pb * DECODE_D + d) = o;
            if (d == 0) {
                part_ml[pb * 2] = gm;
                part_ml[pb * 2 + 1] = gl;
            }
        } else {
            const float inv = gl > 0.f ? 1.f / gl : 0.f;
            *reinterpret_cast<uint2*>(out + row * DECODE_D + d) =
                make_uint2(cvt_pk_bf16(o[0] * inv, o[1] * inv),
                           cvt_pk_bf16(o[2] * inv, o[3] * inv));
        }
    }
}

// out[b, h] = sum_z 2^(m_z - M) acc_z / sum_z 2^(m_z - M) l_z over the splits
// that have keys: 8 splits at a time, 4 dims a thread
__launch_bounds__(256)
__global__ void decode_combine_kernel(
    bf16* __restrict__ out,               // [B, Hq, D]
    const float* __restrict__ part_acc,   // [B, Hq, nsplit, D]
    const float* __restrict__ part_ml,    // [B, Hq, nsplit, 2]
    const int* __restrict__ context_lens, // [B]
    int Hq, int nsplit) {
    const int row = blockIdx.x;  // seq * Hq + head
    const int L = context_lens[row / Hq];
    if (L <= 0) return;
    const int span = span_of(L, nsplit);
    const int used = (L + span - 1) / span;
    const int d = (threadIdx.x & 31) * 4, part = threadIdx.x >> 5;
    const size_t base = (size_t)row * nsplit;
    const float2* ml = reinterpret_cast<const float2*>(part_ml) + base;

    float gm = -INFINITY;
    for (int z = threadIdx.x & 63; z < used; z += 64) gm = fmaxf(gm, ml[z].x);
    gm = wave_reduce_max(gm);
    const float top = gm == -INFINITY ? 0.f : gm;
    float gl = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int z = part; z < used; z += 8) {
        const float2 v = ml[z];
        const float f = __builtin_amdgcn_exp2f(v.x - top);
        gl += f * v.y;
        const f32x4 a = *reinterpret_cast<const f32x4*>(part_acc + (base + z) * DECODE_D + d);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] += f * a[r];
    }
    __shared__ f32x4 o_lds[8][32];
    __shared__ float l_lds[8];
    o_lds[part][threadIdx.x & 31] = o;
    if ((threadIdx.x & 31) == 0) l_lds[part] = gl;
    __syncthreads();
    if (threadIdx.x < 32) {
#pragma unroll
        for (int w = 1; w < 8; ++w) {
            gl += l_lds[w];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] += o_lds[w][threadIdx.x][r];
        }
        const float inv = gl > 0.f ? 1.f / gl : 0.f;
        *reinterpret_cast<uint2*>(out + (size_t)row * DECODE_D + d) = make_uint2(
            cvt_pk_bf16(o[0] * inv, o[1] * inv), cvt_pk_bf16(o[2] * inv, o[3] * inv));
    }
}

extern "C" hipError_t launch_attention_decode(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const float* k_scale, const float* v_scale,
    const int* block_tables, const int* context_lens, float scale, int B,
    int Hq, int Hkv, int block_size, int max_blocks, int D, int64_t q_stride,
    float* part_acc, float* part_ml, int nsplit, hipStream_t stream) {
    if (D != DECODE_D) return hipErrorNotSupported;
    if (Hq % Hkv != 0 || Hq / Hkv > MAX_G) return hipErrorInvalidValue;
    if (nsplit > 1 && (part_acc == nullptr || part_ml == nullptr))
        return hipErrorInvalidValue;
    const int G = Hq / Hkv;
    const bool fp8 = k_scale != nullptr;
    const bool paged = block_size % (fp8 ? 32 : 16) == 0;
    const float scale_log2 = scale * 1.44269504088896f;
    const dim3 grid(B, Hkv, nsplit > 1 ? nsplit : 1);
#define LAUNCH(FP8, SPLIT, PAGED)                                              \
    attention_decode_kernel<FP8, SPLIT, PAGED>                                 \
        <<<grid, dim3(DECODE_WAVES * WAVE_SIZE), 0, stream>>>(                 \
            (bf16*)out, (const bf16*)q, (const char*)k_cache,                  \
            (const char*)v_cache, k_scale, v_scale, block_tables,              \
            context_lens, scale_log2, Hkv, G, block_size, max_blocks,          \
            q_stride, part_acc, part_ml, nsplit)
#define LAUNCH_P(FP8, SPLIT)                                                   \
    do {                                                                       \
        if (paged) LAUNCH(FP8, SPLIT, true);                                   \
        else LAUNCH(FP8, SPLIT, false);                                        \
    } while (0)
    if (fp8 && nsplit > 1) LAUNCH_P(true, true);
    else if (fp8) LAUNCH_P(true, false);
    else if (nsplit > 1) LAUNCH_P(false, true);
    else LAUNCH_P(false, false);
#undef LAUNCH_P
#undef LAUNCH
    HIP_CHECK_LAST();
    if (nsplit > 1) {
        decode_combine_kernel<<<dim3(B * Hq), dim3(256), 0, stream>>>(
            (bf16*)out, part_acc, part_ml, context_lens, Hq, nsplit);
        HIP_CHECK_LAST();
    }
    return hipSuccess;
}
