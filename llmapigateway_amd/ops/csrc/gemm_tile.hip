// Y[M, N] = X[M, K] W[N, K]^T in bf16 for the rows of a batch, up to 256 (in
// parts 512), W as the model holds it.
//
// Up to some 128 rows the read of W bounds it, so a workgroup keeps tiles of depth
// 64 of both operands on their way into LDS, up to 5 of W (direct transfers, one
// barrier a tile), and K is split until there are as many workgroups as CUs. A
// split leaves its part in fp32 for the kernel that reads the product anyway
// (parts_rows.hip): a sum of its own took 4.3 to 5.5 us. Workgroups of one column
// tile start at different depths, so that rows of W at one stride do not all ask
// the same memory channels at once (28672 x 4096: 53 us without, 47.8 with; 128256
// x 4096: 233 and 199); not where the order of sums is asked for, which is that of
// depth then. Above, transfers and products bound it together: 65536 x
// 4096 at 256 rows takes 136 us, its transfers alone 98, its products alone 99.
//
// us, with what reads the parts, against what ran before (the library, tiles over
// a second copy of W in fragment order, or 16-row slabs, each with its reduction):
//                                48 rows       128 rows      256 rows
//   6144 x 4096 and rotation    17.8 (24.1)   22.5 (28.2)   30.8 (33.7)
//   4096 x 4096, addition, norm 14.5 (15.8)   17.1 (19.7)   22.1 (25.6)
//   28672 x 4096 and swiglu     42.8 (52.3)   53.0 (55.1)   68.0 (74.3)
//   4096 x 14336, addition, norm 29.1 (36.5)  34.6 (38.0)   47.2 (51.2)
//   37888 x 3584 and swiglu     49.8 (65.6)   58.8 (81.2)   77.2 (91.2)
//   57344 x 8192 and swiglu      148 (183)     154 (204)     247 (242: kept)
//   128256 x 4096 in fp32        178 (210)     186 (263)     266 (358)

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

namespace {

// all but the last min(TILES, later) tiles of EACH transfers have landed
template <int TILES, int EACH>
__device__ __forceinline__ void wait_all_but(int later) {
    if constexpr (TILES > 0) {
        if (later < TILES) return wait_all_but<TILES - 1, EACH>(later);
    }
    wait_transfers<TILES * EACH>();
}

}  // namespace

// What leaves: the product in fp32, silu(gate) * up of [gate; up] stacked, or a
// split's part of the product in fp32.
enum TileLeaves { TILE_WIDE, TILE_SWIGLU, TILE_PART };

// BM, BN: rows and columns of a workgroup; WM x WN waves share them; NX tiles of
// depth 64 of x and NW of w lie in LDS. Half of the waves fetch x and half w: a
// wave's transfers arrive in order, so one that fetched both would wait for the
// far tiles of w with the near one of x.
template <int BM, int BN, int WM, int WN, int NX, int NW, TileLeaves OUT>
__launch_bounds__(WM* WN* WAVE_SIZE, 2)
__global__ void gemm_tile_kernel(
    void* __restrict__ y, const bf16* __restrict__ x, const bf16* __restrict__ w,
    int M, int N, int K, int n_tiles, int m_tiles, int splits, bool once, bool in_order) {
    constexpr int ROW = 128, F = WM * WN / 2;         // bytes of a tile's row
    constexpr int XB = BM * ROW, WB = BN * ROW;
    constexpr int XMINE = BM / 8 / F, WMINE = BN / 8 / F;  // transfers of 1 KB: 8 rows
    static_assert(BM / 8 % F == 0 && BN / 8 % F == 0 && NX > 1 && NW > 1);
    static_assert((NX - 1) * XMINE < 64 && (NW - 1) * WMINE < 64);
    constexpr int MF = BM / WM / 16, NF = BN / WN / 16;
    static_assert(OUT != TILE_SWIGLU || NF % 2 == 0);
    __shared__ __attribute__((aligned(16))) char lds[NX * XB + NW * WB];

    // the row tiles of a column tile follow each other on one XCD
    const int xcd = blockIdx.x & 7, rest = blockIdx.x >> 3;
    const int m_tile = rest % m_tiles;
    const int n_tile = (rest / m_tiles % ((n_tiles + 7) / 8)) * 8 + xcd;
    const int split = rest / m_tiles / ((n_tiles + 7) / 8);
    if (n_tile >= n_tiles) return;
    const int m0 = m_tile * BM, n0 = n_tile * (OUT == TILE_SWIGLU ? BN / 2 : BN);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;

    const int k_tiles = K / 64;
    const int each = (k_tiles + splits - 1) / splits;
    const int first = split * each, count = max(0, min(k_tiles - first, each));
    const int turn = splits == 1 && count > 0 && !in_order ? (n_tile * 5) % count : 0;

    // this wave's transfers: 8 rows of X or W each; a lane's piece lies so that
    // 16 rows at one piece cover all banks
    const bool fetches_x = wave < F;
    const int mine = (fetches_x ? wave * XMINE : (wave - F) * WMINE) * 8 + (lane >> 3);
    // (from a base that all lanes share: a transfer costs no vector operation)
    const bf16* const base = fetches_x ? x + (int64_t)m0 * K : w + (int64_t)n0 * K;
    constexpr int MINE = XMINE > WMINE ? XMINE : WMINE;
    uint32_t offset[MINE];
#pragma unroll
    for (int j = 0; j < MINE; ++j) {
        const int in = mine + j * 8;
        const int piece = (lane & 7) ^ ((in >> 1) & 7);
        uint32_t row;
        if (fetches_x) {
            row = min(in, M - 1 - m0);
        } else if (OUT == TILE_SWIGLU) {  // blocks of 16: gate, up, gate, up, ..
            row = (in >> 4 & 1) * (N / 2) + min((in >> 5) * 16 + (in & 15), N / 2 - 1 - n0);
        } else {
            row = min(in, N - 1 - n0);
        }
        offset[j] = (row * K + piece * 8) * 2;
    }
    const uint32_t lds_at = __builtin_amdgcn_readfirstlane(
        lds_address(lds) + (fetches_x ? wave * XMINE : (wave - F) * WMINE) * 1024);
    auto k_of = [&](int t) {
        return (int64_t)(first + (t + turn < count ? t + turn : t + turn - count)) * 64;
    };
    auto fetch_x = [&](int t) {
#pragma unroll
        for (int j = 0; j < XMINE; ++j)
            dma16(base + k_of(t), offset[j], lds_at + t % NX * XB + j * 1024);
    };
    auto fetch_w = [&](int t) {
        const bf16* const from = base + k_of(t);
        const uint32_t to = lds_at + NX * XB + t % NW * WB;
        if (once) {
#pragma unroll
            for (int j = 0; j < WMINE; ++j) dma16_once(from, offset[j], to + j * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < WMINE; ++j) dma16(from, offset[j], to + j * 1024);
        }
    };

    f32x4 acc[MF][NF];
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
        for (int n = 0; n < NF; ++n) acc[f][n] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const char* const x_at = lds + (wm * MF * 16 + col) * ROW;
    const char* const w_at = lds + NX * XB + (wn * NF * 16 + col) * ROW;
    bf16x8 xa[MF], wa[NF], xb[MF], wb[NF];
    auto read = [&](bf16x8(&xf)[MF], bf16x8(&wf)[NF], int t, int s) {
        const int piece = ((s * 4 + grp) ^ (col >> 1 & 7)) * 16;
#pragma unroll
        for (int n = 0; n < NF; ++n)
            wf[n] = *reinterpret_cast<const bf16x8*>(w_at + t % NW * WB + n * 16 * ROW + piece);
#pragma unroll
        for (int f = 0; f < MF; ++f)
            xf[f] = *reinterpret_cast<const bf16x8*>(x_at + t % NX * XB + f * 16 * ROW + piece);
    };
    auto multiply = [&](const bf16x8(&xf)[MF], const bf16x8(&wf)[NF]) {
#pragma unroll
        for (int f = 0; f < MF; ++f)
#pragma unroll
            for (int n = 0; n < NF; ++n) acc[f][n] = mfma16(xf[f], wf[n], acc[f][n]);
    };
    // tile t has landed for all waves, and all have read the one before it
    auto arrive = [&](int t) {
        const int later = count - 1 - t;
        if (fetches_x) wait_all_but<NX - 2, XMINE>(later);
        else wait_all_but<NW - 2, WMINE>(later);
        lds_barrier();
    };

    if (count > 0) {
        if (fetches_x) {
#pragma unroll
            for (int t = 0; t < NX - 1; ++t)
                if (t < count) fetch_x(t);
        } else {
#pragma unroll
            for (int t = 0; t < NW - 1; ++t)
                if (t < count) fetch_w(t);
        }
        arrive(0);
        if (fetches_x && NX - 1 < count) fetch_x(NX - 1);
        if (!fetches_x && NW - 1 < count) fetch_w(NW - 1);
        read(xa, wa, 0, 0);
        // a step's fragments are read while the products of the one before
        // run; no branch goes around a read, else the waits that the compiler
        // counts would be for all of them
        auto hold = [&](bf16x8(&xf)[MF], bf16x8(&wf)[NF]) {  // they have arrived
#pragma unroll
            for (int f = 0; f < MF; ++f) asm volatile("" : "+v"(xf[f]));
#pragma unroll
            for (int n = 0; n < NF; ++n) asm volatile("" : "+v"(wf[n]));
        };
        for (int t = 0; t + 1 < count; ++t) {
            read(xb, wb, t, 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(xa, wa);
            __builtin_amdgcn_sched_barrier(0);
            arrive(t + 1);
            hold(xb, wb);
            read(xa, wa, t + 1, 0);
            if (fetches_x && t + NX < count) fetch_x(t + NX);
            if (!fetches_x && t + NW < count) fetch_w(t + NW);
            __builtin_amdgcn_sched_barrier(0);
            multiply(xb, wb);
            __builtin_amdgcn_sched_barrier(0);
        }
        read(xb, wb, count - 1, 1);
        multiply(xa, wa);
        multiply(xb, wb);
    }

#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m0 + wm * MF * 16 + f * 16 + grp * 4 + r;
            if (row >= M) continue;
#pragma unroll
            for (int n = 0; n < NF; n += OUT == TILE_SWIGLU ? 2 : 1) {
                const int c = n0 + (OUT == TILE_SWIGLU ? (wn * NF + n) * 8 : (wn * NF + n) * 16) + col;
                if (c >= (OUT == TILE_SWIGLU ? N / 2 : N)) continue;
                const float v = acc[f][n][r];
                if constexpr (OUT == TILE_SWIGLU)
                    ((bf16*)y)[(int64_t)row * (N / 2) + c] = f2bf(v / (1.f + __expf(-v)) * acc[f][n + 1][r]);
                else if constexpr (OUT == TILE_WIDE)
                    ((float*)y)[(int64_t)row * N + c] = v;
                else
                    ((float*)y)[((int64_t)split * M + row) * N + c] = v;
            }
        }
}

// Tiles of a product in parts. Up to 64 rows tiles have as many, with few columns
// and a short K narrow ones (4096 x 4096 at 48 rows: 10.2 us, 10.9 with 128
// columns), and up to 128 rows two row tiles (13.2 us; 17.1 with 64 x 64; 13.4 with
// 128 x 128, but in 8 parts). Else tiles of 128 x 128, two workgroups a CU whose
// barriers don't meet (128 rows: 14336 deep 28.5 us, 29.4 with one and more tiles
// on their way; 256 rows: 42.9 in 4 parts, 47.7 in 256-row tiles and 8 parts).
// 256-row tiles remain for the largest weights at more than 128 rows, where the
// second row tile's reads show (18944 deep at 160 rows: 44.4 us, 50.2; 12288 x 4096
// at 256: 36.1 and 42.8; 8192 x 28672: 126 and 157).
static int tiles_of(int M, int N, int K, int* bm, int* bn) {
    const bool small = N <= 4608 && K <= 4096;
    const bool large = N > 8192 || (int64_t)N * K > (int64_t)1 << 26;
    *bm = M <= (small ? 128 : 64) ? 64 : M > 128 && large ? 256 : 128;
    *bn = small && M <= 64 ? 64 : 128;
    return (N + *bn - 1) / *bn * ((M + *bm - 1) / *bm);
}
// Splits of K for it: as many workgroups as there are CUs, up to eight a tile;
// twice as many where that leaves a fifth of the CUs without one and two have room
// on a CU (12288 x 4096 at 48 rows: 22.3 us in 5 parts, 28.0 in 2).
extern "C" int gemm_tile_splits(int M, int N, int K) {
    int bm, bn;
    const int tiles = tiles_of(M, N, K, &bm, &bn);
    int s = 256 / tiles;
    if (bm == 64 && M <= 64 && tiles * s < 205) s = 512 / tiles;
    return s < 1 ? 1 : s > 8 ? 8 : s;
}

// leaves: TileLeaves; splits: 1, or with TILE_PART what y has room for; in_order:
// each split's sum by rising depth
extern "C" hipError_t launch_gemm_tile(
    void* y, const void* x, const void* w, int M, int N, int K, int splits, int leaves,
    int in_order, hipStream_t stream) {
    if (M <= 0 || M > (leaves == TILE_PART ? 512 : 256) || N <= 0 || N % 16 != 0 || K <= 0 || K % 64 != 0)
        return hipErrorInvalidValue;
    if ((int64_t)N * K >= (int64_t)1 << 31) return hipErrorInvalidValue;  // 32-bit offsets
    if (leaves == TILE_SWIGLU && N % 32 != 0) return hipErrorInvalidValue;
    if (leaves == TILE_PART ? splits < 1 : splits != 1) return hipErrorInvalidValue;
    const bool once = read_once(N, K);
#define LAUNCH(BM, BN, WM, WN, NX, NW, OUT)                                    \
    do {                                                                       \
        const int n_tiles = (N + BN - 1) / BN, m_tiles = (M + BM - 1) / BM;    \
        const int grid = (n_tiles + 7) / 8 * 8 * m_tiles * splits;             \
        gemm_tile_kernel<BM, BN, WM, WN, NX, NW, OUT>                          \
            <<<grid, dim3(WM * WN * WAVE_SIZE), 0, stream>>>(                  \
                y, (const bf16*)x, (const bf16*)w, M, N, K, n_tiles, m_tiles,  \
                splits, once, in_order != 0);                                                 \
    } while (0)
#define LAUNCH_O(BM, BN, WM, WN, NX, NW)                                       \
    do {                                                                       \
        if (leaves == TILE_SWIGLU) LAUNCH(BM, BN, WM, WN, NX, NW, TILE_SWIGLU);\
        else LAUNCH(BM, BN, WM, WN, NX, NW, TILE_WIDE);                        \
    } while (0)
    int bm, bn;
    tiles_of(M, N, K, &bm, &bn);
    if (leaves == TILE_PART) {
        if (bn == 64) LAUNCH(64, 64, 4, 2, 3, 6, TILE_PART);
        else if (bm == 64 && M > 64) LAUNCH(64, 128, 2, 4, 4, 7, TILE_PART);
        else if (bm == 64) LAUNCH(64, 128, 2, 2, 3, 3, TILE_PART);
        else if (bm == 128) LAUNCH(128, 128, 4, 2, 2, 3, TILE_PART);
        else LAUNCH(256, 128, 4, 4, 3, 4, TILE_PART);
    } else {
        // narrow tiles where 128 columns would leave half of the CUs idle (14336
        // columns at 64 rows: 28.2 us with 64, 35.5 with 128); else one round of
        // workgroups where wider tiles make it one (37888 columns: 53.6 us at 64
        // rows with 192 a tile, 70 with 128)
        const int wide = N <= 16384              ? 64
                         : (N + 127) / 128 <= 256 ? 128
                         : (N + 191) / 192 <= 256 ? 192
                                                  : 256;
        if (wide == 64) {
            if (M <= 128) LAUNCH_O(64, 64, 2, 2, 3, 6);
            else LAUNCH_O(128, 128, 4, 4, 3, 6);
        } else if (M <= 64) {
            if (wide == 128) LAUNCH_O(64, 128, 1, 4, 4, 7);
            else if (wide == 192) LAUNCH_O(64, 192, 2, 2, 3, 5);
            else LAUNCH_O(64, 256, 1, 4, 4, 4);
        } else if (M <= 128) {
            if (wide == 128) LAUNCH_O(128, 128, 4, 4, 3, 6);
            else if (wide == 192) LAUNCH_O(128, 192, 4, 2, 2, 5);
            else LAUNCH_O(128, 256, 2, 4, 2, 4);
        } else {
            if (wide == 192) LAUNCH_O(256, 192, 4, 2, 2, 4);
            else if (wide == 256) LAUNCH_O(256, 256, 4, 2, 2, 3);
            else LAUNCH_O(256, 128, 4, 4, 3, 4);
        }
    }
#undef LAUNCH_O
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}
