// Token sampling for gfx950: greedy argmax / Gumbel-max temperature sampling
// over [B, V] fp32 logits (V up to ~128k). Honors the OpenAI temperature
// param routed through the gateway payload (reference chat.py:116-119).
//
// Two-stage split-V reduction: a single workgroup per sequence leaves 3/4
// of the chip idle at B<=64 and runs latency-bound (measured 160 us for
// 64x128k); stage 1 spreads (B x SPLITS) workgroups over the vocab, stage 2
// combines the per-split winners. Gumbel-max: argmax(logits/T +
// -log(-log(u))) samples softmax(logits/T); noise u comes from the caller
// so CPU and GPU paths share one RNG. 16 bytes a lane, and no noise for what a
// filter has masked: 48 filtered rows of 128256 take 7.6 us instead of 21.6.

#include <type_traits>

#include "common.h"

#define SAMPLE_SPLITS 16

__device__ __forceinline__ void better(
    float v, int i, float& bv, int& bi) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

__launch_bounds__(256)
__global__ void sample_partial_kernel(
    float* __restrict__ part_val,         // [B, SPLITS]
    int* __restrict__ part_idx,           // [B, SPLITS]
    const float* __restrict__ logits,     // [B, V]
    const float* __restrict__ temperature,// [B]
    const float* __restrict__ noise,      // [B, V] or nullptr
    int V) {
    const int b = blockIdx.x;
    const int split = blockIdx.y;
    const int tid = threadIdx.x;
    const float T = temperature[b];
    const bool greedy = (T <= 0.f) || (noise == nullptr);
    const float invT = greedy ? 1.f : 1.f / fmaxf(T, 1e-6f);
    const float* row = logits + (size_t)b * V;
    const float* nrow = noise ? noise + (size_t)b * V : nullptr;

    const int chunk = ((V + SAMPLE_SPLITS - 1) / SAMPLE_SPLITS + 3) / 4 * 4;
    const int lo = min(V, split * chunk);
    const int hi = min(V, lo + chunk);

    float best = -INFINITY;
    int best_idx = lo;
    auto gumbel = [](float u) {
        return -logf(fmaxf(-logf(fmaxf(u, 1e-20f)), 1e-20f));
    };
    // 16 bytes a lane, four loads in flight, where rows allow it
    constexpr int AHEAD = 4;
    const bool wide = V % 4 == 0 && (((uintptr_t)logits | (uintptr_t)noise) & 15) == 0;
    if (wide) {
        for (int i = lo + tid * 4; i < hi; i += AHEAD * 1024) {
            float4 x[AHEAD];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j)
                if (i + j * 1024 < hi) x[j] = *reinterpret_cast<const float4*>(row + i + j * 1024);
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                const int at = i + j * 1024;
                if (at >= hi) continue;
                const float v[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
                if (greedy) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) better(v[e], at + e, best, best_idx);
                    continue;
                }
                // no noise makes -inf win: of a filtered row only what was
                // kept has its noise read
                const bool any = !(v[0] == -INFINITY && v[1] == -INFINITY &&
                                   v[2] == -INFINITY && v[3] == -INFINITY);
                if (!any) continue;
                const float4 u = *reinterpret_cast<const float4*>(nrow + at);
                const float uf[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v[e] != -INFINITY)
                        better(v[e] * invT + gumbel(uf[e]), at + e, best, best_idx);
            }
        }
    } else {
        for (int i = lo + tid; i < hi; i += blockDim.x) {
            float val = row[i];
            if (!greedy) {
                if (val == -INFINITY) continue;
                val = val * invT + gumbel(nrow[i]);
            }
            better(val, i, best, best_idx);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best, off, WAVE_SIZE);
        const int oi = __shfl_xor(best_idx, off, WAVE_SIZE);
        better(ov, oi, best, best_idx);
    }
    __shared__ float sv[4];
    __shared__ int si[4];
    const int wave = tid >> 6;
    if ((tid & 63) == 0) {
        sv[wave] = best;
        si[wave] = best_idx;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int w = 1; w < 4; ++w) better(sv[w], si[w], best, best_idx);
        part_val[b * SAMPLE_SPLITS + split] = best;
        part_idx[b * SAMPLE_SPLITS + split] = best_idx;
    }
}

__launch_bounds__(64)
__global__ void sample_combine_kernel(
    int64_t* __restrict__ out,
    const float* __restrict__ part_val,
    const int* __restrict__ part_idx) {
    const int b = blockIdx.x;
    const int lane = threadIdx.x;
    float v = lane < SAMPLE_SPLITS ? part_val[b * SAMPLE_SPLITS + lane] : -INFINITY;
    int i = lane < SAMPLE_SPLITS ? part_idx[b * SAMPLE_SPLITS + lane] : 0x7FFFFFFF;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        const float ov = __shfl_xor(v, off, WAVE_SIZE);
        const int oi = __shfl_xor(i, off, WAVE_SIZE);
        better(ov, oi, v, i);
    }
    if (lane == 0) out[b] = i;
}

// ---------------------------------------------------------------------------
// top-k / top-p (nucleus) filtering: mask logits outside the kept set to
// -inf, in place, one workgroup per row. No sort: a 2048-bin histogram
// over [max-16, max] locates the coarse threshold bin (counts for top-k,
// exp-mass for top-p), a second 2048-bin histogram WITHIN that bin
// refines the cut to 16/2048^2 ~= 3.8e-6 logit granularity: logits
// closer to the cut than that are kept together (torch's sort breaks
// such ties arbitrarily too).
// Rows with topk[b]==0 and topp[b]>=1 are untouched.
//
// Three passes over the row (513 KB at 128256 tokens) by 16 waves, 16 bytes a
// lane, four loads in flight: maximum; coarse histogram; masking of what lies
// behind the coarse bin, whose own tokens are listed for the fine cut. Bins are
// searched by a scan over the workgroup. 48 rows of 128256 took 607 us by 4
// waves, 4 bytes a lane and one thread's search, 56 so and 41 spread over CUs as
// below; 256 rows 756 and 80. Three quarters are a CU's vector ALU and LDS atomics
// on its row, a quarter latencies that any row pays (32000 tokens take 25 us).
// ---------------------------------------------------------------------------

#define TPF_BINS 2048
#define TPF_RANGE 16.0f  // logits below max-16 carry < 1.2e-7 of the mass
#define TPF_THREADS 1024
#define TPF_WAVES (TPF_THREADS / WAVE_SIZE)
#define TPF_LIST 4096  // of a coarse bin's tokens, as a rule tens

// A softmax mass relative to the row's largest, e in [0, 1], as a multiple of
// 1 / units (mass_units below; at most 2^42, so that the low half of a double
// that is 2^52 more has it). Sums of these do not depend on their order, and are
// as close as fp32 sums at least: up to 2^20 tokens round to 2^-43 each, 128256 of
// them to 1.5e-8 together if all do so one way. LDS adds whole numbers in one
// instruction (fp32 in a loop of compare-and-swap: 190 us a row). A NaN is none.
__device__ __forceinline__ unsigned long long mass_of(float e, double units) {
    return __double_as_longlong(fma((double)fmaxf(e, 0.f), units, 0x1p52)) & ((1ull << 52) - 1);
}
// 2^42, or what the sum over V tokens leaves room for
static double mass_units(int V) {
    double units = 0x1p42;
    for (int64_t most = 1 << 20; most < V; most *= 2) units /= 2;
    return units;
}

// f(value, its index) over a row of V floats, whose start need not be aligned
// to 16 bytes; WRITE stores what f left
template <bool WRITE, typename F>
__device__ __forceinline__ void for_row(float* row, int V, F f) {
    const int tid = threadIdx.x;
    const int head = min(V, (int)((16 - ((uintptr_t)row & 15)) & 15) / 4);
    if (tid < head) {
        float v = row[tid];
        if (f(v, tid) && WRITE) row[tid] = v;
    }
    const int n4 = (V - head) / 4;
    float4* body = reinterpret_cast<float4*>(row + head);
    constexpr int AHEAD = 4;
    for (int i = tid; i < n4; i += AHEAD * TPF_THREADS) {
        float4 v[AHEAD];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (i + j * TPF_THREADS < n4) v[j] = body[i + j * TPF_THREADS];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const int p = i + j * TPF_THREADS, at = head + p * 4;
            if (p >= n4) continue;
            bool changed = f(v[j].x, at);
            changed |= f(v[j].y, at + 1);
            changed |= f(v[j].z, at + 2);
            changed |= f(v[j].w, at + 3);
            if (WRITE && changed) body[p] = v[j];
        }
    }
    const int done = head + n4 * 4;
    if (tid < V - done) {
        float v = row[done + tid];
        if (f(v, done + tid) && WRITE) row[done + tid] = v;
    }
}

// The first of ``bins`` bins at which the running count or mass reaches its
// need, and both sums in front of it; -1 where none does. For all threads.
struct Crossing {
    int bin, count;
    unsigned long long mass;
};
__device__ __forceinline__ Crossing find_crossing(
    const int* cnt, const unsigned long long* mass, int bins, int count0,
    unsigned long long mass0, unsigned long long need_mass, long long need_count) {
    constexpr int EACH = TPF_BINS / TPF_THREADS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ int w_cnt[TPF_WAVES];
    __shared__ unsigned long long w_mass[TPF_WAVES];
    __shared__ int found;
    __shared__ Crossing out;
    int c = 0;
    unsigned long long m = 0;
#pragma unroll
    for (int j = 0; j < EACH; ++j) {
        c += cnt[tid * EACH + j];
        m += mass[tid * EACH + j];
    }
    int ci = c;
    unsigned long long mi = m;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int oc = __shfl_up(ci, off, 64);
        const unsigned long long om = __shfl_up(mi, off, 64);
        if (lane >= off) {
            ci += oc;
            mi += om;
        }
    }
    if (lane == 63) {
        w_cnt[wave] = ci;
        w_mass[wave] = mi;
    }
    if (tid == 0) found = TPF_BINS;
    __syncthreads();
    int count = count0;
    unsigned long long total = mass0;
#pragma unroll
    for (int w = 0; w < TPF_WAVES; ++w) {  // (all read at once)
        const int wc = w_cnt[w];
        const unsigned long long wm = w_mass[w];
        if (w < wave) {
            count += wc;
            total += wm;
        }
    }
    count += ci - c;
    total += mi - m;
    int mine = TPF_BINS;
    Crossing at{-1, 0, 0};
#pragma unroll
    for (int j = 0; j < EACH; ++j) {
        const int bin = tid * EACH + j;
        const int before = count;
        const unsigned long long above = total;
        count += cnt[bin];
        total += mass[bin];
        if (mine == TPF_BINS && bin < bins && (total >= need_mass || count >= need_count)) {
            mine = bin;
            at = {bin, before, above};
        }
    }
    if (mine < TPF_BINS) atomicMin(&found, mine);
    __syncthreads();
    if (mine < TPF_BINS && found == mine) out = at;
    if (found == TPF_BINS && tid == 0) out = {-1, 0, 0};
    __syncthreads();
    return out;
}

#define TPF_SCALE (TPF_BINS / TPF_RANGE)

// bin of a distance d >= 0 from the largest; +inf-safe (masked rows)
__device__ __forceinline__ int coarse_bin(float d) {
    return min((int)(d * TPF_SCALE), TPF_BINS - 1);
}

__device__ __forceinline__ unsigned long long block_sum(
    unsigned long long z, unsigned long long* sums) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) z += __shfl_xor(z, off, WAVE_SIZE);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = z;
    __syncthreads();
    z = 0;
#pragma unroll
    for (int w = 0; w < TPF_WAVES; ++w) z += sums[w];
    return z;
}

// the histogram of V values; returns, for a wave, NaN with any mass that is
__device__ __forceinline__ float coarse_histogram(
    float* row, int V, float m, double units, bool do_k, bool do_p, int* cnt,
    unsigned long long* mass) {
    float nan = 0.f;
    auto histogram = [&](auto with_count, auto with_mass) {
        for_row<false>(row, V, [&](float& x, int) {
            const float d = m - x;
            const int bin = coarse_bin(d);
            if constexpr (with_count.value) atomicAdd(&cnt[bin], 1);
            if constexpr (with_mass.value) {
                const float e = __expf(-d);
                nan += e;
                atomicAdd(&mass[bin], mass_of(e, units));
            }
            return false;
        });
    };
    if (!do_p) histogram(std::true_type(), std::false_type());
    else if (!do_k) histogram(std::false_type(), std::true_type());
    else histogram(std::true_type(), std::true_type());
    return wave_reduce_sum(nan);
}

// no mass is enough where there is a NaN
__device__ __forceinline__ unsigned long long mass_needed(
    bool do_p, float nan, float p, unsigned long long z) {
    return do_p && nan == nan ? (unsigned long long)ceil(fmax((double)p, 0.0) * (double)z) : ~0ull;
}

__device__ __forceinline__ void fine_count(
    float d, int coarse, double units, bool do_k, bool do_p, int* cnt,
    unsigned long long* mass) {
    const float d_lo = coarse / TPF_SCALE;  // the bin's lower edge (distance)
    const int fine = max(0, min((int)((d - d_lo) * (TPF_SCALE * TPF_BINS)), TPF_BINS - 1));
    if (do_k) atomicAdd(&cnt[fine], 1);
    if (do_p) atomicAdd(&mass[fine], mass_of(__expf(-d), units));
}

// distances strictly below the fine bin's upper edge are kept
__device__ __forceinline__ float fine_cut(int coarse, const Crossing& fine) {
    const int last = fine.bin < 0 ? TPF_BINS - 1 : fine.bin;
    return coarse / TPF_SCALE + (last + 1) / (TPF_SCALE * TPF_BINS);
}

// the coarse bin's own: by the list, or by the row if there are more
__device__ __forceinline__ void mask_behind(
    float* row, int V, const int* list, int listed, float m, float d_cut) {
    auto mask = [&](float& x, int) {
        if (!(m - x >= d_cut)) return false;
        x = -INFINITY;
        return true;
    };
    if (listed <= TPF_LIST) {
        for (int i = threadIdx.x; i < listed; i += TPF_THREADS) {
            float x = row[list[i]];
            if (mask(x, 0)) row[list[i]] = x;
        }
    } else {
        for_row<true>(row, V, mask);
    }
}

__device__ __forceinline__ float block_max(float m, float* red) {
    m = wave_reduce_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < TPF_WAVES; ++w) m = fmaxf(m, red[w]);
    return m;
}

__launch_bounds__(TPF_THREADS)
__global__ void topk_topp_filter_kernel(
    float* __restrict__ logits,          // [B, V], filtered in place
    const float* __restrict__ topp,      // [B]; >= 1 disables
    const int* __restrict__ topk,        // [B]; 0 disables
    int V, double units) {
    const int b = blockIdx.x;
    const float p = topp[b];
    const int k = topk[b];
    const bool do_p = p < 1.0f;
    const bool do_k = k > 0;
    if (!do_p && !do_k) return;
    float* row = logits + (size_t)b * V;
    const int tid = threadIdx.x;

    __shared__ float s_red[TPF_WAVES], s_nan[TPF_WAVES];
    __shared__ unsigned long long s_sum[TPF_WAVES];
    __shared__ int s_cnt[TPF_BINS];
    __shared__ unsigned long long s_mass[TPF_BINS];
    __shared__ int s_listed, s_list[TPF_LIST];

    // ---- pass 1: row max ----
    float m = -INFINITY;
    for_row<false>(row, V, [&](float& x, int) {
        m = fmaxf(m, x);
        return false;
    });
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        s_cnt[i] = 0;
        s_mass[i] = 0;
    }
    if (tid == 0) s_listed = 0;
    m = block_max(m, s_red);

    // ---- pass 2: coarse histogram ----
    float nan = coarse_histogram(row, V, m, units, do_k, do_p, s_cnt, s_mass);
    if ((tid & 63) == 0) s_nan[tid >> 6] = nan;
    __syncthreads();  // bins complete
    unsigned long long z = 0;  // all mass
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) z += s_mass[i];
    z = block_sum(z, s_sum);
    nan = 0.f;
#pragma unroll
    for (int w = 0; w < TPF_WAVES; ++w) nan += s_nan[w];

    const unsigned long long need_mass = mass_needed(do_p, nan, p, z);
    const long long need_count = do_k ? k : 0x7FFFFFFFLL;
    // a crossing in the last bin, which has the tail: everything is kept
    const Crossing coarse =
        find_crossing(s_cnt, s_mass, TPF_BINS - 1, 0, 0, need_mass, need_count);
    if (coarse.bin < 0) return;

    // ---- pass 3: mask behind the coarse bin, fine histogram within it ----
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        s_cnt[i] = 0;
        s_mass[i] = 0;
    }
    __syncthreads();
    for_row<true>(row, V, [&](float& x, int at) {
        const float d = m - x;
        const int bin = coarse_bin(d);  // of a NaN 0, in front of or in every other
        if (bin < coarse.bin) return false;
        if (bin == coarse.bin) {
            fine_count(d, coarse.bin, units, do_k, do_p, s_cnt, s_mass);
            const int n = atomicAdd(&s_listed, 1);
            if (n < TPF_LIST) s_list[n] = at;
            return false;
        }
        x = -INFINITY;
        return true;
    });
    __syncthreads();
    const Crossing fine = find_crossing(
        s_cnt, s_mass, TPF_BINS, coarse.count, coarse.mass, need_mass, need_count);
    mask_behind(row, V, s_list, s_listed, m, fine_cut(coarse.bin, fine));
}

// ---------------------------------------------------------------------------
// The same with a row spread over several workgroups, where rows alone leave CUs
// idle: maxima of the pieces; their coarse histograms; masking behind the coarse
// bin, whose tokens are listed; the fine cut by one workgroup a row. Masses are
// whole numbers, so that the cut is the one above to the last token.
// ---------------------------------------------------------------------------

struct FilterRow {  // what a row's last kernel takes from the one before
    float most;
    int bin, count;
    unsigned long long mass, need_mass;
};
struct FilterPieces {
    unsigned long long* mass;  // [B, TPF_BINS]
    int* cnt;                  // [B, TPF_BINS]
    float* most;               // [B, pieces]
    float* nan;                // [B, pieces]
    FilterRow* row;            // [B]
    int* listed;               // [B]
    int* list;                 // [B, TPF_LIST]
    int pieces, V;
    double units;

    __device__ __forceinline__ int first(int piece) const {
        const int each = ((V + pieces - 1) / pieces + 3) / 4 * 4;
        return min(V, piece * each);
    }
};

__launch_bounds__(TPF_THREADS)
__global__ void filter_max_kernel(
    float* __restrict__ logits, const float* __restrict__ topp, const int* __restrict__ topk,
    FilterPieces f) {
    const int b = blockIdx.x, piece = blockIdx.y;
    if (topp[b] >= 1.0f && topk[b] <= 0) return;
    __shared__ float red[TPF_WAVES];
    for (int i = piece * TPF_THREADS + threadIdx.x; i < TPF_BINS; i += f.pieces * TPF_THREADS) {
        f.mass[(size_t)b * TPF_BINS + i] = 0;
        f.cnt[(size_t)b * TPF_BINS + i] = 0;
    }
    const int lo = f.first(piece);
    float m = -INFINITY;
    for_row<false>(logits + (size_t)b * f.V + lo, f.first(piece + 1) - lo, [&](float& x, int) {
        m = fmaxf(m, x);
        return false;
    });
    m = block_max(m, red);
    if (threadIdx.x == 0) {
        f.most[b * f.pieces + piece] = m;
        if (piece == 0) f.listed[b] = 0;
    }
}

__launch_bounds__(TPF_THREADS)
__global__ void filter_coarse_kernel(
    float* __restrict__ logits, const float* __restrict__ topp, const int* __restrict__ topk,
    FilterPieces f) {
    const int b = blockIdx.x, piece = blockIdx.y, tid = threadIdx.x;
    const bool do_p = topp[b] < 1.0f, do_k = topk[b] > 0;
    if (!do_p && !do_k) return;
    __shared__ float s_red[TPF_WAVES];
    __shared__ int s_cnt[TPF_BINS];
    __shared__ unsigned long long s_mass[TPF_BINS];
    float m = -INFINITY;
    for (int i = 0; i < f.pieces; ++i) m = fmaxf(m, f.most[b * f.pieces + i]);
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        s_cnt[i] = 0;
        s_mass[i] = 0;
    }
    __syncthreads();
    const int lo = f.first(piece);
    const float nan = coarse_histogram(
        logits + (size_t)b * f.V + lo, f.first(piece + 1) - lo, m, f.units, do_k, do_p, s_cnt,
        s_mass);
    if ((tid & 63) == 0) s_red[tid >> 6] = nan;
    __syncthreads();
    const size_t at = (size_t)b * TPF_BINS;
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        if (do_k && s_cnt[i] != 0) atomicAdd(&f.cnt[at + i], s_cnt[i]);
        if (do_p && s_mass[i] != 0) atomicAdd(&f.mass[at + i], s_mass[i]);
    }
    if (tid == 0) {
        float sum = 0.f;
        for (int w = 0; w < TPF_WAVES; ++w) sum += s_red[w];
        f.nan[b * f.pieces + piece] = sum;
    }
}

__launch_bounds__(TPF_THREADS)
__global__ void filter_mask_kernel(
    float* __restrict__ logits, const float* __restrict__ topp, const int* __restrict__ topk,
    FilterPieces f) {
    const int b = blockIdx.x, piece = blockIdx.y, tid = threadIdx.x;
    const float p = topp[b];
    const int k = topk[b];
    const bool do_p = p < 1.0f, do_k = k > 0;
    if (!do_p && !do_k) return;
    __shared__ unsigned long long s_sum[TPF_WAVES];
    __shared__ int s_cnt[TPF_BINS];
    __shared__ unsigned long long s_mass[TPF_BINS];
    __shared__ int s_listed, s_base, s_list[TPF_LIST];
    float m = -INFINITY, nan = 0.f;
    for (int i = 0; i < f.pieces; ++i) {
        m = fmaxf(m, f.most[b * f.pieces + i]);
        nan += f.nan[b * f.pieces + i];
    }
    unsigned long long z = 0;  // all mass
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        s_cnt[i] = f.cnt[(size_t)b * TPF_BINS + i];
        z += s_mass[i] = f.mass[(size_t)b * TPF_BINS + i];
    }
    if (tid == 0) s_listed = 0;
    z = block_sum(z, s_sum);
    const unsigned long long need_mass = mass_needed(do_p, nan, p, z);
    const Crossing coarse = find_crossing(
        s_cnt, s_mass, TPF_BINS - 1, 0, 0, need_mass, do_k ? k : 0x7FFFFFFFLL);
    if (piece == 0 && tid == 0)
        f.row[b] = {m, coarse.bin, coarse.count, coarse.mass, need_mass};
    if (coarse.bin < 0) return;

    const int lo = f.first(piece);
    for_row<true>(logits + (size_t)b * f.V + lo, f.first(piece + 1) - lo, [&](float& x, int at) {
        const int bin = coarse_bin(m - x);
        if (bin < coarse.bin) return false;
        if (bin == coarse.bin) {
            const int n = atomicAdd(&s_listed, 1);
            if (n < TPF_LIST) s_list[n] = lo + at;
            return false;
        }
        x = -INFINITY;
        return true;
    });
    __syncthreads();
    if (tid == 0) s_base = atomicAdd(&f.listed[b], s_listed);
    __syncthreads();
    for (int i = tid; i < min(s_listed, TPF_LIST) && s_base + i < TPF_LIST; i += TPF_THREADS)
        f.list[(size_t)b * TPF_LIST + s_base + i] = s_list[i];
}

__launch_bounds__(TPF_THREADS)
__global__ void filter_fine_kernel(
    float* __restrict__ logits, const float* __restrict__ topp, const int* __restrict__ topk,
    FilterPieces f) {
    const int b = blockIdx.x, tid = threadIdx.x;
    const int k = topk[b];
    const bool do_p = topp[b] < 1.0f, do_k = k > 0;
    if (!do_p && !do_k) return;
    const FilterRow r = f.row[b];
    if (r.bin < 0) return;
    __shared__ int s_cnt[TPF_BINS];
    __shared__ unsigned long long s_mass[TPF_BINS];
    for (int i = tid; i < TPF_BINS; i += TPF_THREADS) {
        s_cnt[i] = 0;
        s_mass[i] = 0;
    }
    __syncthreads();
    float* row = logits + (size_t)b * f.V;
    const int* list = f.list + (size_t)b * TPF_LIST;
    const int listed = f.listed[b];
    auto count = [&](float& x, int) {
        const float d = r.most - x;
        if (coarse_bin(d) == r.bin) fine_count(d, r.bin, f.units, do_k, do_p, s_cnt, s_mass);
        return false;
    };
    if (listed <= TPF_LIST) {
        for (int i = tid; i < listed; i += TPF_THREADS) count(row[list[i]], 0);
    } else {
        for_row<false>(row, f.V, count);
    }
    __syncthreads();
    const Crossing fine = find_crossing(
        s_cnt, s_mass, TPF_BINS, r.count, r.mass, r.need_mass, do_k ? k : 0x7FFFFFFFLL);
    mask_behind(row, f.V, list, listed, r.most, fine_cut(r.bin, fine));
}

// Workgroups that a row is spread over: as many as let all rows fill the 256 CUs,
// where that makes up for three more launches (128256 tokens: 1 row 26.5 us, 50 by
// one workgroup, 48 rows 41 and 56, 64 rows 45 and 57, 85 rows in 3 pieces 52 and
// 55, 128 in 2 70 and 71; 64000 tokens: 1 row 25.5 and 29, 48 rows 35 and 33).
static int filter_pieces(int B, int V) {
    return V >= 3 << 15 && B > 0 && B <= 64 ? min(256 / B, 16) : 1;
}
extern "C" size_t filter_scratch_bytes(int B, int V) {
    const int pieces = filter_pieces(B, V);
    if (pieces == 1) return 0;
    return (size_t)B * (TPF_BINS * 12 + pieces * 8 + sizeof(FilterRow) + 4 + TPF_LIST * 4);
}

// scratch: filter_scratch_bytes, aligned to 8
extern "C" hipError_t launch_topk_topp_filter(
    float* logits, const float* topp, const int* topk, int B, int V, void* scratch,
    hipStream_t stream) {
    const int pieces = filter_pieces(B, V);
    if (pieces == 1) {
        topk_topp_filter_kernel<<<B, TPF_THREADS, 0, stream>>>(
            logits, topp, topk, V, mass_units(V));
        HIP_CHECK_LAST();
        return hipSuccess;
    }
    FilterPieces f;
    const size_t n = (size_t)B * pieces;
    f.mass = (unsigned long long*)scratch;
    f.row = (FilterRow*)(f.mass + (size_t)B * TPF_BINS);
    f.cnt = (int*)(f.row + B);
    f.most = (float*)(f.cnt + (size_t)B * TPF_BINS);
    f.nan = f.most + n;
    f.listed = (int*)(f.nan + n);
    f.list = f.listed + B;
    f.pieces = pieces;
    f.V = V;
    f.units = mass_units(V);
    const dim3 grid(B, pieces);
    filter_max_kernel<<<grid, TPF_THREADS, 0, stream>>>(logits, topp, topk, f);
    HIP_CHECK_LAST();
    filter_coarse_kernel<<<grid, TPF_THREADS, 0, stream>>>(logits, topp, topk, f);
    HIP_CHECK_LAST();
    filter_mask_kernel<<<grid, TPF_THREADS, 0, stream>>>(logits, topp, topk, f);
    HIP_CHECK_LAST();
    filter_fine_kernel<<<B, TPF_THREADS, 0, stream>>>(logits, topp, topk, f);
    HIP_CHECK_LAST();
    return hipSuccess;
}

extern "C" hipError_t launch_sample(
    int64_t* out, const float* logits, const float* temperature,
    const float* noise, float* part_val, int* part_idx, int B, int V,
    hipStream_t stream) {
    dim3 grid1(B, SAMPLE_SPLITS);
    sample_partial_kernel<<<grid1, 256, 0, stream>>>(
        part_val, part_idx, logits, temperature, noise, V);
    HIP_CHECK_LAST();
    sample_combine_kernel<<<B, 64, 0, stream>>>(out, part_val, part_idx);
    HIP_CHECK_LAST();
    return hipSuccess;
}
