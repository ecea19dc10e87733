// Y[M, N] = X[M, K] W[N, K]^T in bf16 for few rows (decode steps, short
// prompts), bound by the one reading of W, which lies as the model holds it.
//
// - A workgroup has 16 to 64 output columns (16 NF) and all of K; its waves
//   share K, tile by tile in turn, so sums meet in LDS inside the workgroup and
//   not in slabs of memory behind a second kernel.
// - Each wave streams its tiles of W and X (rows of 128 or 256 bytes in a
//   piece) through a ring of two in LDS by transfers that need no registers,
//   waited for by count; no barrier before the sums meet. Rings of 53 to 82 KB
//   let two workgroups share a CU; those of eight waves (115 to 147 KB), where
//   there are no more workgroups than CUs, and of 32 rows 128 deep (98 KB) have
//   one to themselves.
// - A decode step's small kernels are part of the products beside them, as each
//   alone is a launch of 5-6 us: the RMS norm in front (x enters times the
//   norm's weights, rounded as the normed row is; its rows' squares are summed
//   on the way and scale the sums), the addition to the stream behind, the
//   rotation and page writes of queries, keys and values. What an epilogue
//   reads for that comes by transfers too, since a wait for a load would be a
//   wait for every tile.
// - SWIGLU: W is [gate; up] stacked, a workgroup has as many columns of each, a
//   block of either or two in every wave, and silu(gate) * up leaves it; the
//   product is never written. Rotated heads are alike, 16 columns of the first
//   half beside those of the second. Tiles of 64 there: x, its norm and the wave's
//   turn serve two blocks (28672 x 4096 with norm, 16 rows: 41.4 us; blocks in
//   waves of their own, 128 deep: 46.6; 6144 x 4096 with rotation 15.1 and 16.3).
//   Products of one block gain nothing by that (128256 x 4096: 181 us and 154).
//
// What bounds it is the memory's rate for large W (128256 x 4096 at one row:
// 155 us, 6.8 TB/s) and launch, first tile and sums (3-4 us) for small; from 32
// rows on also the rows of X, which every workgroup reads. us by rows, W cold,
// "was" with the slab kernel or the macro tile:
//                        1 row          16            32
//    6144 x 4096      17.3 -> 11.2  19.8 -> 12.9  (library 15.5, stays)
//    4096 x 4096      10.4 ->  8.5  15.0 ->  8.8  15.3 -> 10.6
//    4096 x 14336     30.8 -> 21.5  38.2 -> 24.9  38.4 -> 30.6
//   28672 x 4096, and
//     its swiglu     53.7 -> 39.5  65.5 -> 41.4  66.0 -> 46.4
//   37888 x 3584,
//     the same       59.7 -> 44.5  61.8 -> 46.0  62.5 -> 53.8

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

// What leaves a product: itself, in bf16 or fp32; silu(gate) * up of [gate; up]
// stacked; its sum with what y holds; the rotated query, key and value rows,
// which also go to their pages.
enum Leaves { PLAIN, SWIGLU, ADD, WIDE, ROTATED };

struct StreamArgs {
    void* y;        // [M, N], or [M, N / 2] (SWIGLU); fp32 (WIDE)
    const bf16* x;  // [M, K]
    const bf16* w;  // [N, K]
    int M, N, K;
    bool once;         // w is read past the caches
    const bf16* norm;  // [K]: x enters as RMS norm of its rows (NORM)
    float eps;
    // ROTATED: N is (Hq + 2 Hkv) * D
    const int64_t* positions;  // [M]
    const float* cos_sin;      // [positions, D]: cosines, sines
    const int64_t* slots;      // [M], -1: no page
    bf16* k_cache;             // [pages, Hkv, block_size, D]
    bf16* v_cache;
    int Hq, Hkv, D, block_size;
};

// MT, NF: blocks of 16 rows and of 16 columns; W: waves; KT: depth of a tile.
template <int MT, int NF, int W, int KT, Leaves OUT, bool NORM>
__launch_bounds__(W* WAVE_SIZE)
__global__ void gemm_stream_kernel(const StreamArgs a) {
    const int M = a.M, N = a.N, K = a.K;
    constexpr int ROW = KT * 2;             // bytes of a row of a tile
    constexpr int PIECES = ROW / 16;
    constexpr int ROWS = 1024 / ROW;        // of a transfer
    constexpr int MOVES = 16 / ROWS;        // of a block of 16 rows
    constexpr int BLOCKS = NF + MT, IN_FLIGHT = BLOCKS * MOVES + (NORM ? 1 : 0);
    constexpr int SLOT = BLOCKS * 16 * ROW + (NORM ? 1024 : 0);
    // 16 rows at one piece cover all banks once (two rows share them at 64)
    auto place = [](int row, int piece) { return piece ^ (KT == 64 ? (row >> 1) & 7 : row & 15); };

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int subs = OUT == ROTATED ? a.D / 32 : 1;  // blocks of half a head
    const int head = OUT == ROTATED ? blockIdx.x / subs : 0;
    const int n0 = OUT == ROTATED ? head * a.D + blockIdx.x % subs * 16
                                  : blockIdx.x * (OUT == SWIGLU ? NF * 8 : NF * 16);
    // the second half of the column blocks: up's, or what is rotated with the first
    constexpr bool PAIRS = OUT == SWIGLU || OUT == ROTATED;
    static_assert(!PAIRS || NF % 2 == 0);
    static_assert(OUT != ROTATED || NF == 2);
    const int to_pair = OUT == ROTATED ? a.D / 2 : N / 2;

    __shared__ __attribute__((aligned(16))) char ring[W][2][SLOT];
    const uint32_t ring_at = __builtin_amdgcn_readfirstlane(lds_address(&ring[wave][0][0]));

    // a lane's part of a transfer: row ROWS*j + lane/PIECES, the piece whose
    // place its 16 bytes of LDS are
    const int t_row = lane / PIECES, t_piece = lane % PIECES;
    uint32_t w_off[MOVES], x_off[MT][MOVES];
#pragma unroll
    for (int j = 0; j < MOVES; ++j) {
        const int r = j * ROWS + t_row;
        w_off[j] = ((uint32_t)r * K + place(r, t_piece) * 8) * 2;
#pragma unroll
        for (int f = 0; f < MT; ++f)
            x_off[f][j] = ((uint32_t)min(f * 16 + r, M - 1) * K + place(r, t_piece) * 8) * 2;
    }
    const bf16* w_block[NF];
#pragma unroll
    for (int n = 0; n < NF; ++n)
        w_block[n] = a.w + (int64_t)(PAIRS && n >= NF / 2 ? to_pair + n0 + (n - NF / 2) * 16
                                                          : n0 + n * 16) * K;

    // what the epilogue takes besides, brought by wave 0 while the tiles come:
    // the sums' other part, or positions and slots and then their angles
    __shared__ __attribute__((aligned(16))) bf16 held[OUT == ADD ? MT * 16 : 1][16];
    __shared__ int64_t of_row[OUT == ROTATED ? 2 : 1][32];
    __shared__ float turn[OUT == ROTATED ? 2 : 1][OUT == ROTATED ? MT * 16 : 1][16];

    const int tiles = (K + KT - 1) / KT;
    const int mine = wave < tiles ? (tiles - wave + W - 1) / W : 0;
    auto fetch = [&](int i) {
        const int k0 = (wave + i * W) * KT;
        const uint32_t at = ring_at + (i & 1) * SLOT;
        // the slot's last fragments have left it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // behind the end of a row: its first piece, which no product takes
        const bool part = k0 + KT > K;
#pragma unroll
        for (int j = 0; j < MOVES; ++j) {
            const uint32_t back =
                part && k0 + place(j * ROWS + t_row, t_piece) * 8 >= K
                    ? place(j * ROWS + t_row, t_piece) * 16 : 0;
            if (a.once) {
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    dma16_once(w_block[n] + k0, w_off[j] - back, at + (n * MOVES + j) * 1024);
            } else {
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    dma16(w_block[n] + k0, w_off[j] - back, at + (n * MOVES + j) * 1024);
            }
#pragma unroll
            for (int f = 0; f < MT; ++f)
                dma16(a.x + k0, x_off[f][j] - back, at + ((NF + f) * MOVES + j) * 1024);
        }
        if (NORM) {  // one row of the norm's weights (ROWS times the same)
            const uint32_t off = part && k0 + t_piece * 8 >= K ? 0 : t_piece * 16;
            dma16(a.norm + k0, off, at + BLOCKS * 16 * ROW);
        }
    };

    f32x4 acc[MT][NF];
#pragma unroll
    for (int f = 0; f < MT; ++f)
#pragma unroll
        for (int n = 0; n < NF; ++n) acc[f][n] = (f32x4){0.f, 0.f, 0.f, 0.f};

    float squares[MT];  // of row col, this lane's depths
#pragma unroll
    for (int f = 0; f < MT; ++f) squares[f] = 0.f;

    if (OUT == ADD && wave == 0) {  // 8 rows of 32 bytes a transfer
#pragma unroll
        for (int j = 0; j < MT * 2; ++j)
            dma4(reinterpret_cast<const float*>(
                     (const bf16*)a.y + (int64_t)min(j * 8 + lane / 8, M - 1) * N + n0) + lane % 8,
                 __builtin_amdgcn_readfirstlane(lds_address(&held[j * 8][0])));
    }
    if (OUT == ROTATED && wave == 0) {  // up to 32 rows of 8 bytes
        const int at = min(lane, 2 * M - 1);
        dma4(reinterpret_cast<const float*>(a.positions) + at,
             __builtin_amdgcn_readfirstlane(lds_address(&of_row[0][0])));
        dma4(reinterpret_cast<const float*>(a.slots) + at,
             __builtin_amdgcn_readfirstlane(lds_address(&of_row[1][0])));
    }
    if (mine > 0) fetch(0);
    if (mine > 1) fetch(1);
    if (OUT == ROTATED && wave == 0) {
        if (mine > 1) wait_transfers<2 * IN_FLIGHT>();
        else if (mine > 0) wait_transfers<IN_FLIGHT>();
        else wait_transfers<0>();
#pragma unroll
        for (int j = 0; j < MT * 4; ++j) {  // 4 rows of 16 columns
            const int64_t position = of_row[0][min(j * 4 + grp, M - 1)];
            const float* cs = a.cos_sin + position * a.D + n0 % a.D + col;
            dma4(cs, __builtin_amdgcn_readfirstlane(lds_address(&turn[0][j * 4][0])));
            dma4(cs + a.D / 2, __builtin_amdgcn_readfirstlane(lds_address(&turn[1][j * 4][0])));
        }
    }
    // (a wave that brings more only waits longer for its first tile)
    for (int i = 0; i < mine; ++i) {
        if (i + 1 < mine) wait_transfers<IN_FLIGHT>();
        else wait_transfers<0>();
        const char* tile = ring[wave][i & 1];
        const int k0 = (wave + i * W) * KT;
#pragma unroll
        for (int s = 0; s < KT / 32; ++s) {
            if (k0 + s * 32 >= K) break;
            const int at = col * ROW + place(col, s * 4 + grp) * 16;
            bf16x8 xf[MT];
#pragma unroll
            for (int f = 0; f < MT; ++f)
                xf[f] = *reinterpret_cast<const bf16x8*>(tile + (NF + f) * 16 * ROW + at);
            if (NORM) {
                float g[8];
                unpack8(*reinterpret_cast<const uint4*>(tile + BLOCKS * 16 * ROW + (s * 4 + grp) * 16), g);
#pragma unroll
                for (int f = 0; f < MT; ++f) {
                    float v[8];
                    unpack8(*reinterpret_cast<const uint4*>(&xf[f]), v);
#pragma unroll
                    for (int j = 0; j < 8; ++j) squares[f] = fmaf(v[j], v[j], squares[f]);
                    xf[f] = as_frag(make_uint4(
                        cvt_pk_bf16(v[0] * g[0], v[1] * g[1]), cvt_pk_bf16(v[2] * g[2], v[3] * g[3]),
                        cvt_pk_bf16(v[4] * g[4], v[5] * g[5]), cvt_pk_bf16(v[6] * g[6], v[7] * g[7])));
                }
            }
#pragma unroll
            for (int n = 0; n < NF; ++n) {
                const bf16x8 wf = *reinterpret_cast<const bf16x8*>(tile + n * 16 * ROW + at);
#pragma unroll
                for (int f = 0; f < MT; ++f) acc[f][n] = mfma16(xf[f], wf, acc[f][n]);
            }
        }
        if (i + 2 < mine) fetch(i + 2);
    }
    if (OUT == ADD || OUT == ROTATED) wait_transfers<0>();  // of a wave without tiles

    __shared__ float square_sums[NORM ? W : 1][MT * 16];
    if (NORM) {
#pragma unroll
        for (int f = 0; f < MT; ++f) {
            float v = squares[f];
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (grp == 0) square_sums[wave][f * 16 + col] = v;
        }
    }

    // ---- the waves' sums meet, half of them into the other half ----
    static_assert(W / 2 * MT * NF * 1024 <= W * 2 * SLOT);
    __syncthreads();  // all tiles read
    f32x4* sums = reinterpret_cast<f32x4*>(&ring[0][0][0]);
#pragma unroll
    for (int h = W / 2; h > 0; h >>= 1) {
        if (wave >= h && wave < 2 * h) {
#pragma unroll
            for (int f = 0; f < MT; ++f)
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    sums[(((wave - h) * MT + f) * NF + n) * 64 + lane] = acc[f][n];
        }
        __syncthreads();
        if (wave < h) {
#pragma unroll
            for (int f = 0; f < MT; ++f)
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    acc[f][n] += sums[((wave * MT + f) * NF + n) * 64 + lane];
        }
        __syncthreads();
    }
    if (wave != 0) return;
#pragma unroll
    for (int f = 0; f < MT; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = f * 16 + grp * 4 + r;
            if (row >= M) continue;
            float by = 1.f;
            if (NORM) {
                float q = 0.f;
#pragma unroll
                for (int p = 0; p < W; ++p) q += square_sums[p][row];
                by = rsqrtf(q / K + a.eps);
            }
            bf16* out = (bf16*)a.y + (int64_t)row * (OUT == SWIGLU ? N / 2 : N) + n0 + col;
            if constexpr (OUT == WIDE) {
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    ((float*)a.y)[(int64_t)row * N + n0 + col + n * 16] = acc[f][n][r] * by;
            } else if constexpr (OUT == ROTATED) {
                float lo = acc[f][0][r] * by, hi = acc[f][1][r] * by;
                if (head < a.Hq + a.Hkv) {
                    const float c = turn[0][row][col], s = turn[1][row][col];
                    const float v = lo * c - hi * s;
                    hi = hi * c + lo * s;
                    lo = v;
                }
                out[0] = f2bf(lo);
                out[to_pair] = f2bf(hi);
                const int64_t slot = of_row[1][row];
                if (head >= a.Hq && slot >= 0) {
                    bf16* cache = head < a.Hq + a.Hkv ? a.k_cache : a.v_cache;
                    const int64_t at = ((slot / a.block_size) * a.Hkv + (head - a.Hq) % a.Hkv) *
                                           a.block_size + slot % a.block_size;
                    cache[at * a.D + n0 % a.D + col] = f2bf(lo);
                    cache[at * a.D + n0 % a.D + col + to_pair] = f2bf(hi);
                }
            } else {
#pragma unroll
                for (int n = 0; n < (OUT == SWIGLU ? NF / 2 : NF); ++n) {
                    float v = acc[f][n][r] * by;
                    if (OUT == SWIGLU) v = v / (1.f + __expf(-v)) * acc[f][n + NF / 2][r] * by;
                    if (OUT == ADD) v += bf2f(held[row][col]);
                    out[n * 16] = f2bf(v);
                }
            }
        }
}

// For 1 to 64 rows (swiglu: 48; addition and rotation: 32; with norm: 32, or 16
// without a swiglu or rotation behind; fp32: 16, without norm, which in front of a
// head's many columns costs more than a kernel: 172 us and 155 + 3); columns in
// 16s (swiglu: N in 64s; rotation: head sizes in 32s), K in 32s, rows of x, w
// and norm aligned to 16 bytes, K below 2^25.
static hipError_t launch_stream(StreamArgs a, Leaves out, hipStream_t stream) {
    a.once = read_once(a.N, a.K);
    const int M = a.M, N = a.N, K = a.K;
    const bool norm = a.norm != nullptr;
    const int most = out == WIDE || (out == PLAIN && norm) ? 16
                     : norm || out >= ADD                  ? 32
                     : out == SWIGLU                       ? 48 : 64;
    if (M <= 0 || M > most || K <= 0 || K % 32 != 0 || K >= (1 << 25)) return hipErrorInvalidValue;
    if (N <= 0 || N % (out == SWIGLU ? 64 : 16) != 0) return hipErrorInvalidValue;
    if (out == ROTATED && (!norm || a.D % 32 != 0 || a.block_size <= 0 || a.Hkv <= 0 ||
                           (a.Hq + 2 * a.Hkv) * a.D != N))
        return hipErrorInvalidValue;
    if ((out == ADD || out == WIDE) && norm) return hipErrorInvalidValue;
#define LAUNCH(MT, NF, W, KT, OUT, NORM)                                       \
    gemm_stream_kernel<MT, NF, W, KT, OUT, NORM>                               \
        <<<N / (NF * 16), \
           dim3(W * WAVE_SIZE), 0, stream>>>(a)
#define LAUNCH_N(MT, NF, W, KT, OUT)                                           \
    do {                                                                       \
        if (norm) LAUNCH(MT, NF, W, KT, OUT, true);                            \
        else LAUNCH(MT, NF, W, KT, OUT, false);                                \
    } while (0)
    // one workgroup a CU at most: more waves there
    const bool few = N / 16 <= 256;
    if (out == ROTATED) {
        if (M <= 16 && N / 32 <= 256) LAUNCH(1, 2, 8, 64, ROTATED, true);
        else if (M <= 16) LAUNCH(1, 2, 4, 64, ROTATED, true);
        else if (N / 32 <= 256) LAUNCH(2, 2, 8, 64, ROTATED, true);
        else LAUNCH(2, 2, 4, 64, ROTATED, true);
    } else if (out == SWIGLU) {
        if (M <= 16) LAUNCH_N(1, 2, 4, 64, SWIGLU);
        else if (M <= 32) LAUNCH_N(2, 4, 2, 64, SWIGLU);
        else LAUNCH(3, 4, 2, 64, SWIGLU, false);
    } else if (out == ADD) {
        if (M > 16) LAUNCH(2, 1, 4, 128, ADD, false);
        else if (few) LAUNCH(1, 1, 8, 128, ADD, false);
        else LAUNCH(1, 1, 4, 128, ADD, false);
    } else if (out == WIDE) {
        LAUNCH(1, 1, 4, 128, WIDE, false);
    } else if (M <= 16) {
        if (few && !norm) LAUNCH(1, 1, 8, 128, PLAIN, false);
        else LAUNCH_N(1, 1, 4, 128, PLAIN);
    } else if (M <= 32) {
        LAUNCH(2, 1, 4, 128, PLAIN, false);
    } else if (M <= 48) {
        LAUNCH(3, 1, 4, 64, PLAIN, false);
    } else {
        LAUNCH(4, 1, 4, 64, PLAIN, false);
    }
#undef LAUNCH_N
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}

// leaves: 0 the product, 1 swiglu of it, 2 its sum with y, 3 the product in fp32;
// norm may be null
extern "C" hipError_t launch_gemm_stream(
    void* y, const void* x, const void* w, int M, int N, int K, int leaves, const void* norm,
    float eps, hipStream_t stream) {
    if (leaves < PLAIN || leaves > WIDE) return hipErrorInvalidValue;
    StreamArgs a{};
    a.y = y;
    a.x = (const bf16*)x;
    a.w = (const bf16*)w;
    a.M = M;
    a.N = N;
    a.K = K;
    a.norm = (const bf16*)norm;
    a.eps = eps;
    return launch_stream(a, (Leaves)leaves, stream);
}

extern "C" hipError_t launch_gemm_stream_qkv(
    void* y, const void* x, const void* w, int M, int K, const void* norm, float eps,
    const int64_t* positions, const float* cos_sin, const int64_t* slots, void* k_cache,
    void* v_cache, int Hq, int Hkv, int D, int block_size, hipStream_t stream) {
    StreamArgs a{};
    a.y = y;
    a.x = (const bf16*)x;
    a.w = (const bf16*)w;
    a.M = M;
    a.N = (Hq + 2 * Hkv) * D;
    a.K = K;
    a.norm = (const bf16*)norm;
    a.eps = eps;
    a.positions = positions;
    a.cos_sin = cos_sin;
    a.slots = slots;
    a.k_cache = (bf16*)k_cache;
    a.v_cache = (bf16*)v_cache;
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.D = D;
    a.block_size = block_size;
    return launch_stream(a, ROTATED, stream);
}
