// What reads a product that lies in parts, fp32 [splits, T, N] (gemm_tile.hip):
// adding them up is part of the step's next small kernel instead of a kernel of
// its own, and the sums keep their fp32 until the result is rounded once.
//
// Latency bounds both: a launch, one round trip to memory for all parts at once,
// and for the norm one more for its sum; from some 100 rows the read of the parts,
// at 6 TB/s. 64 rows of 4096 in 8 parts, added and normed: 3.7 us with 1024 threads
// a row, 5.0 with 256; 256 rows 7.7 and 8.6. 64 rows of 6144 in 5 parts, rotated:
// 3 us. As kernels of their own the sums took 4.3 to 5.5 us, the norm 5.4 to 9.9,
// rotation and page writes 6.4 to 9.

#include "common.h"
#include <hip/hip_fp8.h>
#include "mfma.h"

__device__ __forceinline__ f32x4 unpack4(uint2 u) {
    return (f32x4){__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                   __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
}
__device__ __forceinline__ uint2 pack4(f32x4 f) {
    return make_uint2(cvt_pk_bf16(f[0], f[1]), cvt_pk_bf16(f[2], f[3]));
}

// r += sum of parts; out = rmsnorm(r) * weight. A workgroup of THREADS has a row,
// a thread CHUNKS pieces of 4 columns, whose parts are all on their way at once.
template <int THREADS, int CHUNKS>
__launch_bounds__(THREADS)
__global__ void add_parts_norm_kernel(
    bf16* __restrict__ out,           // [T, H]
    bf16* __restrict__ r,             // [T, H]
    const float* __restrict__ parts,  // [splits, T, H]
    const bf16* __restrict__ weight,  // [H]
    float eps, int T, int H, int splits) {
    const int row = blockIdx.x, tid = threadIdx.x;
    f32x4 v[CHUNKS];
    uint2 was[CHUNKS], g[CHUNKS];
    float squares = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int at = (tid + c * THREADS) * 4;
        if (at >= H) continue;
        was[c] = *reinterpret_cast<const uint2*>(r + (int64_t)row * H + at);
        g[c] = *reinterpret_cast<const uint2*>(weight + at);
        const float* p = parts + (int64_t)row * H + at;
        v[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int s = 0; s < splits; ++s)
            v[c] += *reinterpret_cast<const f32x4*>(p + (int64_t)s * T * H);
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int at = (tid + c * THREADS) * 4;
        if (at >= H) continue;
        const uint2 sum = pack4(v[c] + unpack4(was[c]));
        *reinterpret_cast<uint2*>(r + (int64_t)row * H + at) = sum;
        v[c] = unpack4(sum);  // the norm is that of the stored row
#pragma unroll
        for (int j = 0; j < 4; ++j) squares = fmaf(v[c][j], v[c][j], squares);
    }
    __shared__ float red[THREADS / WAVE_SIZE];
    squares = wave_reduce_sum(squares);
    if ((tid & 63) == 0) red[tid >> 6] = squares;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < THREADS / WAVE_SIZE; ++w) total += red[w];
    const float inv = rsqrtf(total / H + eps);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int at = (tid + c * THREADS) * 4;
        if (at >= H) continue;
        *reinterpret_cast<uint2*>(out + (int64_t)row * H + at) =
            pack4(v[c] * inv * unpack4(g[c]));
    }
}

extern "C" hipError_t launch_add_parts_norm(
    void* out, void* r, const float* parts, const void* weight, float eps, int T, int H,
    int splits, hipStream_t stream) {
    if (T <= 0 || H <= 0 || H % 8 != 0 || H > 16384 || splits < 1)
        return hipErrorInvalidValue;
#define LAUNCH(THREADS, C)                                                     \
    add_parts_norm_kernel<THREADS, C><<<T, THREADS, 0, stream>>>(              \
        (bf16*)out, (bf16*)r, parts, (const bf16*)weight, eps, T, H, splits)
    // (a row of 4096 by 1024 threads 3.1 us, by 256 with 16 columns each 5.2)
    if (H <= 1024) LAUNCH(256, 1);
    else if (H <= 2048) LAUNCH(512, 1);
    else if (H <= 4096) LAUNCH(1024, 1);
    else if (H <= 8192) LAUNCH(1024, 2);
    else LAUNCH(1024, 4);
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}

// r = the tokens' rows of the embedding; out, if given, = rmsnorm(r) * weight. As
// above; 3 us where a gather takes 4 to 11 and a norm behind it 4.
template <int THREADS, int CHUNKS>
__launch_bounds__(THREADS)
__global__ void embed_norm_kernel(
    bf16* __restrict__ out,            // [T, H] or null
    bf16* __restrict__ r,              // [T, H]
    const int64_t* __restrict__ tokens,  // [T]
    const bf16* __restrict__ embed,    // [V, H]
    const bf16* __restrict__ weight,   // [H]
    float eps, int64_t V, int H) {
    const int row = blockIdx.x, tid = threadIdx.x;
    const int64_t token = tokens[row];
    const bool known = token >= 0 && token < V;
    f32x4 v[CHUNKS];
    uint2 g[CHUNKS];
    float squares = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int at = (tid + c * THREADS) * 4;
        if (at >= H) continue;
        // a token that the embedding does not have: NaN
        uint2 x = make_uint2(0x7fc07fc0u, 0x7fc07fc0u);
        if (known) x = *reinterpret_cast<const uint2*>(embed + token * H + at);
        if (out != nullptr) g[c] = *reinterpret_cast<const uint2*>(weight + at);
        *reinterpret_cast<uint2*>(r + (int64_t)row * H + at) = x;
        v[c] = unpack4(x);
#pragma unroll
        for (int j = 0; j < 4; ++j) squares = fmaf(v[c][j], v[c][j], squares);
    }
    if (out == nullptr) return;
    __shared__ float red[THREADS / WAVE_SIZE];
    squares = wave_reduce_sum(squares);
    if ((tid & 63) == 0) red[tid >> 6] = squares;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < THREADS / WAVE_SIZE; ++w) total += red[w];
    const float inv = rsqrtf(total / H + eps);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int at = (tid + c * THREADS) * 4;
        if (at >= H) continue;
        *reinterpret_cast<uint2*>(out + (int64_t)row * H + at) =
            pack4(v[c] * inv * unpack4(g[c]));
    }
}

extern "C" hipError_t launch_embed_norm(
    void* out, void* r, const int64_t* tokens, const void* embed, const void* weight, float eps,
    int T, int64_t V, int H, hipStream_t stream) {
    if (T <= 0 || V <= 0 || H <= 0 || H % 8 != 0 || H > 16384) return hipErrorInvalidValue;
#define LAUNCH(THREADS, C)                                                     \
    embed_norm_kernel<THREADS, C><<<T, THREADS, 0, stream>>>(                  \
        (bf16*)out, (bf16*)r, tokens, (const bf16*)embed, (const bf16*)weight, eps, V, H)
    if (H <= 1024) LAUNCH(256, 1);
    else if (H <= 2048) LAUNCH(512, 1);
    else if (H <= 4096) LAUNCH(1024, 1);
    else if (H <= 8192) LAUNCH(1024, 2);
    else LAUNCH(1024, 4);
#undef LAUNCH
    HIP_CHECK_LAST();
    return hipSuccess;
}

#define PARTS_THREADS 256

// Rows of query, key and value heads of 128 from their parts: the first two
// rotated, keys and values also into their pages, in bf16 or e4m3 with a scale a
// row. A wave has a head of a row, a lane the pair of columns that rotate.
template <bool FP8>
__launch_bounds__(PARTS_THREADS)
__global__ void rotate_parts_kernel(
    bf16* __restrict__ y,                     // [T, (Hq + 2 Hkv) * 128]
    const float* __restrict__ parts,          // [splits, T, the same]
    const int64_t* __restrict__ positions,    // [T]
    const float* __restrict__ cos_sin,        // [positions, 128]
    const int64_t* __restrict__ slots,        // [T], -1: no page
    void* __restrict__ k_cache, void* __restrict__ v_cache,  // [NB, Hkv, BS, 128]
    float* __restrict__ k_scale, float* __restrict__ v_scale,
    int T, int Hq, int Hkv, int block_size, int splits) {
    constexpr int D = 128, HALF = 64;
    const int row = blockIdx.x, lane = threadIdx.x & 63;
    const int heads = Hq + 2 * Hkv;
    const int head = blockIdx.y * (PARTS_THREADS / WAVE_SIZE) + (threadIdx.x >> 6);
    if (head >= heads) return;
    const int64_t at = ((int64_t)row * heads + head) * D + lane;
    const float* cs = cos_sin + positions[row] * D;
    const float c = cs[lane], s = cs[HALF + lane];
    float lo = 0.f, hi = 0.f;
#pragma unroll 8
    for (int p = 0; p < splits; ++p) {
        lo += parts[at + (int64_t)p * T * heads * D];
        hi += parts[at + (int64_t)p * T * heads * D + HALF];
    }
    if (head < Hq + Hkv) {
        const float a = lo * c - hi * s;
        hi = hi * c + lo * s;
        lo = a;
    }
    const bf16 lo_b = f2bf(lo), hi_b = f2bf(hi);
    y[at] = lo_b;
    y[at + HALF] = hi_b;
    const int64_t slot = slots[row];
    if (head < Hq || slot < 0) return;
    const bool is_k = head < Hq + Hkv;
    const int64_t to =
        ((slot / block_size) * Hkv + (head - Hq) % Hkv) * block_size + slot % block_size;
    if constexpr (FP8) {
        lo = bf2f(lo_b);  // as a row in bf16 is quantized
        hi = bf2f(hi_b);
        const float top = wave_reduce_max(fmaxf(fabsf(lo), fabsf(hi)));
        const float scale = top > 0.f ? top / FP8_MAX : 1.f;
        if (lane == 0) (is_k ? k_scale : v_scale)[to] = scale;
        unsigned char* cache = (unsigned char*)(is_k ? k_cache : v_cache) + to * D;
        cache[lane] = f2fp8(lo / scale);
        cache[HALF + lane] = f2fp8(hi / scale);
    } else {
        bf16* cache = (bf16*)(is_k ? k_cache : v_cache) + to * D;
        cache[lane] = lo_b;
        cache[HALF + lane] = hi_b;
    }
}

extern "C" hipError_t launch_rotate_parts(
    void* y, const float* parts, const int64_t* positions, const float* cos_sin,
    const int64_t* slots, void* k_cache, void* v_cache, float* k_scale, float* v_scale, int T,
    int Hq, int Hkv, int block_size, int splits, hipStream_t stream) {
    if (T <= 0 || Hq <= 0 || Hkv <= 0 || block_size <= 0 || splits < 1)
        return hipErrorInvalidValue;
    const dim3 grid(T, (Hq + 2 * Hkv + 3) / 4);
    if (k_scale != nullptr)
        rotate_parts_kernel<true><<<grid, PARTS_THREADS, 0, stream>>>(
            (bf16*)y, parts, positions, cos_sin, slots, k_cache, v_cache, k_scale, v_scale, T,
            Hq, Hkv, block_size, splits);
    else
        rotate_parts_kernel<false><<<grid, PARTS_THREADS, 0, stream>>>(
            (bf16*)y, parts, positions, cos_sin, slots, k_cache, v_cache, nullptr, nullptr, T,
            Hq, Hkv, block_size, splits);
    HIP_CHECK_LAST();
    return hipSuccess;
}
