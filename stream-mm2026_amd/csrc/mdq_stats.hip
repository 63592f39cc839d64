// mdq_stats.hip -- per-tensor gradient statistics of the MDQ bit decision,
// for a whole tensor list in two launches.
//
// The reference computes, per tensor and before the step (stquant_opt_simple.py:93-98),
//   n_l = sqrt(mean(g^2)),  r_l = std(g) / (mean(|g|) + 1e-12),  v_l = mean(g^2)
// with std unbiased, as separate fp32 torch reductions per tensor.  Here:
//   1. stats_partial_kernel: one 512-thread workgroup per 32768-element tile of
//      one tensor writes four fp64 partials: sum g, M2 = sum (g - tile mean)^2,
//      sum g^2 (fp32 squares, as the reference's grad * grad) and sum |g|.
//      Each thread loads its 64 elements with 16-byte loads and sums x, x^2 and |x|
//      over each load pairwise in fp32 (at most 3 roundings, 1.8e-7 of the summed
//      magnitudes), and these short sums across loads in fp64.  Near the HBM
//      roofline the kernel is close to VALU-bound (about ten lane instructions per
//      element fit in the memory time); this path takes about seven.  The thread's M2 comes from sum x^2 - (sum x)^2 / 64
//      where that cancellation loses at most a bit; where the mean dominates the
//      spread the registers are summed again as deviations from the thread's fp32
//      mean, and non-finite or tiny (squares below fp32's normal range) values are
//      redone in fp64.  The threads' (mean, M2) then merge pairwise by Chan's
//      formula for equal counts, across lanes and across the workgroup's waves.
//      A ragged last tile, and every tile of a tensor that does not start on 16 bytes (a
//      view of a flat grad buffer), takes per-element fp64 sums and a second pass for the
//      deviations from its mean: thread i sums the elements i, i + 512, ... in that order,
//      so the bits do not depend on where in its line the tensor starts (tile_f64).  About
//      twenty lane operations an element, twelve of them fp64 or conversions: 16-bit views
//      are VALU-bound there (257 ragged bf16 tensors packed back to back, 726 MB: 184 us a
//      call, 119 on 16-byte boundaries), fp32 views near the memory's rate (1453 MB: 234 us).
//      Loaded one element at a time, each waited for, they took 700 and 732 us.
//   2. stats_finish_kernel: one workgroup per tensor combines its tiles in a fixed
//      order.  The squared deviations combine by Chan's pairwise formula,
//      M2 = sum M2_i + sum n_i (mean_i - mean)^2, which stays accurate however
//      large |mean| is against the spread.  The results are rounded to the
//      reference's fp32 outputs.  A sum whose exact value exceeds FLT_MAX gives
//      inf, as the reference's fp32 accumulators overflow.
//   3. scores_kernel (a call of its own, after the caller's mean over the tensors):
//      one thread per tensor folds the mean into the EMAs and forms the tensor's score.
// Both orders are fixed by the tensors' sizes and by whether each starts on 16 bytes, so results
// are deterministic and do not depend on the addresses otherwise.
#include <hip/hip_runtime.h>

#include "mdq_desc.h"
#include "mdq_stats.h"

namespace mdq {

namespace {

constexpr int ST_THREADS = 512;
constexpr int ST_WAVES = ST_THREADS / 64;

__device__ __forceinline__ float bf16_to_f(uint32_t h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ float f16_to_f(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// The grads' pointers come from the descriptor table, so the compiler cannot tell
// they are global memory: without the cast it emits flat loads, which it can only
// wait for all together.
#define ST_GLOBAL __attribute__((address_space(1)))

// Element e of a grad at any byte address: the element types below ask for no alignment, which
// costs nothing (a load of 2 or 4 bytes is one instruction at any address on this target).
typedef float any_f32 __attribute__((aligned(1)));
typedef unsigned short any_u16 __attribute__((aligned(1)));

template <int GT>
__device__ __forceinline__ float load_one(const void *g, int64_t e)
{
    if constexpr (GT == GT_F32) return ((const ST_GLOBAL any_f32 *)g)[e];
    else if constexpr (GT == GT_BF16) return bf16_to_f(((const ST_GLOBAL any_u16 *)g)[e]);
    else return f16_to_f(((const ST_GLOBAL any_u16 *)g)[e]);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Elements per 16-byte load.
template <int GT> constexpr int vec_elems() { return GT == GT_F32 ? 4 : 8; }

// One 16-byte non-temporal load at element e (16-byte aligned), kept as loaded
// (16-bit grads take half the registers of their fp32 values).
template <int GT>
__device__ __forceinline__ u32x4 load_raw(const void *g, int64_t e)
{
    constexpr int ES = GT == GT_F32 ? 4 : 2;   // bytes per element
    return __builtin_nontemporal_load((const ST_GLOBAL u32x4 *)(static_cast<const char *>(g) + ES * e));
}

// The fp32 values of one loaded 16-byte vector.
template <int GT>
__device__ __forceinline__ void widen(const u32x4 v, float (&x)[vec_elems<GT>()])
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    if constexpr (GT == GT_F32) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = __uint_as_float(w[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[2 * k] = GT == GT_BF16 ? bf16_to_f(w[k] & 0xffffu) : f16_to_f(w[k] & 0xffffu);
            x[2 * k + 1] = GT == GT_BF16 ? bf16_to_f(w[k] >> 16) : f16_to_f(w[k] >> 16);
        }
    }
}

// fp64 sums of one element: g, g^2 (the fp32 square), |g|
__device__ __forceinline__ void acc(double &s1, double &s2, double &sa, float x)
{
    s1 += (double)x;
    s2 += (double)(x * x);
    sa += fabs((double)x);
}

// Pairwise fp32 sum of N = 4 or 8 values.
template <int N>
__device__ __forceinline__ float pair_sum(const float (&x)[N])
{
    const float a = (x[0] + x[1]) + (x[2] + x[3]);
    if constexpr (N == 4) return a;
    else return a + ((x[4] + x[5]) + (x[6] + x[7]));
}

// Chan et al.'s merge of two disjoint parts of n elements each into (mean, M2) of
// their union: mean = (mean_a + mean_b) / 2, M2 = M2_a + M2_b + (n / 2) delta^2.
// Symmetric in the two parts, bit for bit, so both lanes of a butterfly exchange
// hold the same result.
__device__ __forceinline__ void merge_equal(double &mean, double &m2, double om, double om2, int n)
{
    const double dl = om - mean;
    m2 = fma(dl, dl * (0.5 * n), m2 + om2);
    mean = (mean + om) * 0.5;
}

// Sum of K doubles over the workgroup; the totals are returned in every thread
// (through LDS), summed in a fixed order.
template <int K>
__device__ __forceinline__ void block_sum(double (&v)[K], double (*lds)[K])
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] += __shfl_xor(v[k], off, 64);
    const int w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) lds[w][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double t = lds[0][k];
#pragma unroll
        for (int q = 1; q < ST_WAVES; ++q) t += lds[q][k];
        v[k] = t;
    }
    __syncthreads();   // lds is free for the next block_sum
}

// The partial sums of a tile of cnt elements from per-element fp64 sums: the tile mean, then the
// squared deviations from it.  each(f) calls f(value, whether it is one of the tile's) for this
// thread's elements i, i + 512, ... in that order.
template <class Each>
__device__ __forceinline__ void tile_f64(uint32_t cnt, Each each, double *__restrict__ partial, double (*lds3)[3],
                                         double (*lds2)[2])
{
    double s[3] = {0.0, 0.0, 0.0};      // sum g, sum g^2, sum |g|
    each([&](float x, bool in) { acc(s[0], s[1], s[2], in ? x : 0.0f); });
    block_sum<3>(s, lds3);
    const double n_t = (double)cnt;
    const float c = (float)(s[0] / n_t);
    double dv[2] = {0.0, 0.0};          // sum d, sum d^2 with d = g - c
    each([&](float x, bool in) {
        const double dd = in ? (double)x - (double)c : 0.0;
        dv[0] += dd;
        dv[1] = fma(dd, dd, dv[1]);
    });
    block_sum<2>(dv, lds2);
    if (threadIdx.x == 0) {
        // d = g - c is exact in fp64, so M2 = sum d^2 - (sum d)^2 / n and sum g = n c + sum d
        // are as accurate as the tile's spread allows (non-finite g: the first pass's sum)
        partial[0] = fabs(dv[0]) <= __DBL_MAX__ ? fma(n_t, (double)c, dv[0]) : s[0];
        partial[1] = dv[1] - dv[0] * (dv[0] / n_t);
        partial[2] = s[1];
        partial[3] = s[2];
    }
}

// A whole tile at any byte address.  Each thread keeps its elements from the first pass for the
// second (a 16-bit pair in one register), 113 registers in fp32 and 85-88 in 16 bits; read again
// instead, 8 in flight as for a ragged tile, the 257 ragged tensors take 350 us in place of 234 in
// fp32 and 227 in place of 184 in bf16.  16 loads at a time: 32 and 64 take 196 and 203 us in bf16.
template <int GT>
__device__ __forceinline__ void whole_f64(const void *g, double *__restrict__ partial, double (*lds3)[3],
                                          double (*lds2)[2])
{
    constexpr int NE = STAT_TILE / ST_THREADS;     // elements per thread
    constexpr int P = GT == GT_F32 ? 1 : 2;        // elements per register
    constexpr int G = 16;                          // loaded together
    uint32_t raw[NE / P];
#pragma unroll
    for (int k0 = 0; k0 < NE; k0 += G) {
        uint32_t w[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint32_t i = (uint32_t)((k0 + k) * ST_THREADS) + threadIdx.x;
            if constexpr (P == 1) w[k] = __float_as_uint(((const ST_GLOBAL any_f32 *)g)[i]);
            else w[k] = ((const ST_GLOBAL any_u16 *)g)[i];
        }
#pragma unroll
        for (int k = 0; k < G; k += P) raw[(k0 + k) / P] = P == 1 ? w[k] : w[k] | (w[k + P - 1] << 16);
    }
    tile_f64((uint32_t)STAT_TILE, [&](auto &&f) {
#pragma unroll
        for (int r = 0; r < NE / P; ++r) {
            // opaque in each pass: the compiler would keep every element's fp64 value from the
            // first one, 128 registers, instead of widening it again
            asm volatile("" : "+v"(raw[r]));
            if constexpr (GT == GT_F32) {
                f(__uint_as_float(raw[r]), true);
            } else {
                f(GT == GT_BF16 ? bf16_to_f(raw[r] & 0xffffu) : f16_to_f(raw[r] & 0xffffu), true);
                f(GT == GT_BF16 ? bf16_to_f(raw[r] >> 16) : f16_to_f(raw[r] >> 16), true);
            }
        }
    }, partial, lds3, lds2);
}

// A ragged last tile of cnt elements at any byte address, read once a pass (the second time from
// L2) with 16 loads a thread in flight: 24 spill at 6 waves per SIMD, 8 run 100 ragged tensors in
// 24.5 us in place of 23.9.
template <int GT>
__device__ __forceinline__ void ragged_f64(const void *g, uint32_t cnt, double *__restrict__ partial, double (*lds3)[3],
                                           double (*lds2)[2])
{
    constexpr int G = 16;
    tile_f64(cnt, [&](auto &&f) {
#pragma unroll 1
        for (uint32_t i0 = threadIdx.x; i0 < cnt; i0 += G * ST_THREADS) {
            float x[G];
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const uint32_t i = i0 + (uint32_t)(k * ST_THREADS);
                x[k] = load_one<GT>(g, i < cnt ? i : cnt - 1u);
            }
#pragma unroll
            for (int k = 0; k < G; ++k) f(x[k], i0 + (uint32_t)(k * ST_THREADS) < cnt);
        }
    }, partial, lds3, lds2);
}

// OFF16: some tensor of the launch starts off 16 bytes and has a whole tile.  An instance of its
// own: whole_f64's registers would leave the 16-byte path 4 waves per SIMD (257 aligned ragged
// bf16 tensors 119 -> 135 us).  The counts are asked for: left to itself the compiler gives the
// other instance 84 registers and 5 waves, and this one's loads less room (199 us in place of 191).
template <int GT, bool OFF16>
__global__ __launch_bounds__(ST_THREADS) __attribute__((amdgpu_waves_per_eu(OFF16 ? 4 : 6)))
void stats_partial_kernel(const StatDesc *__restrict__ d, int n, const long long *__restrict__ tb,
                          double *__restrict__ partials)
{
    __shared__ double lds4[ST_WAVES][4];
    __shared__ double lds3[ST_WAVES][3];
    __shared__ double lds2[ST_WAVES][2];
    // Workgroup b runs on XCD x = b % 8 as its j-th (j = b / 8); the tiles go to
    // the XCDs in round-robin chunks of 16 (2^19 elements), the workgroups of the
    // last, partial round of 8 chunks take tile b (a bijection on [0, grid)).
    // LLaMA-7B bf16 grads, same-allocation A/B: 1.89 ms against 2.00 ms for
    // tile = b; chunks of 32-128 tiles run as 16.
    constexpr unsigned CK = 16u;
    const unsigned grid = gridDim.x, b = blockIdx.x, j = b >> 3, x = b & 7u;
    const long long tile = b < grid / (8u * CK) * (8u * CK) ? (long long)((j / CK) * 8u + x) * CK + (j % CK)
                                                            : (long long)b;
    // the tensor owning this tile: the last i with tile_begin[i] <= tile
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tb[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    const StatDesc t = d[lo];
    const int64_t base = (tile - t.tile_begin) * STAT_TILE;
    const int64_t left = t.numel - base;           // elements from the tile's first one on
    if (left >= STAT_TILE && (!OFF16 || (reinterpret_cast<uintptr_t>(t.g) % 16) == 0)) {
        // One pass: each thread loads its STAT_TILE / ST_THREADS elements and sums x,
        // x^2 and |x| (fp32 over each loaded group, pairwise; fp64 across groups).
        constexpr int V = vec_elems<GT>();
        constexpr int NL = STAT_TILE / (V * ST_THREADS);
        constexpr double NT = (double)(V * NL);        // elements per thread
        u32x4 raw[NL];
#pragma unroll
        for (int k = 0; k < NL; ++k) raw[k] = load_raw<GT>(t.g, base + V * ((int64_t)k * ST_THREADS + threadIdx.x));
        // the element in place e of this thread's load k
        const auto pos = [&](int k, int e) { return base + V * ((int64_t)k * ST_THREADS + threadIdx.x) + e; };
        double sx = 0.0, sq = 0.0, ab = 0.0;
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            float x[V], x2[V], xa[V];
            widen<GT>(raw[k], x);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                x2[e] = x[e] * x[e];
                xa[e] = fabsf(x[e]);
            }
            sx += (double)pair_sum<V>(x);
            sq += (double)pair_sum<V>(x2);
            ab += (double)pair_sum<V>(xa);
        }
        // The thread's M2 = sum x^2 - (sum x)^2 / n loses at most one bit to cancellation
        // where (sum x)^2 / n <= sum x^2 / 2, i.e. the mean is not large against the spread
        // (zero-mean-like gradients).  Elsewhere the registers are summed again as
        // deviations from the fp32 thread mean (exact where x is within a factor 2 of it);
        // non-finite sums (a non-finite x, or fp32 sums beyond FLT_MAX) and values so small
        // that fp32 squares lose bits (mean |x| or mean |x - mean| below 2^-60) are redone
        // in fp64 from memory.
        double mean = sx * (1.0 / NT);
        double m2 = fma(-sx, mean, sq);
        bool exact = fabs(sx) <= __DBL_MAX__ && sq <= __DBL_MAX__ && !(ab > 0.0 && ab < 0x1p-60 * NT);
        if (exact && !(sx * sx <= 0.5 * NT * sq)) {
            const float c = (float)mean;
            double s1 = 0.0, s2 = 0.0, sd = 0.0;
#pragma unroll
            for (int k = 0; k < NL; ++k) {
                float x[V], dv[V], d2[V], da[V];
                widen<GT>(raw[k], x);
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    dv[e] = x[e] - c;
                    d2[e] = dv[e] * dv[e];
                    da[e] = fabsf(dv[e]);
                }
                s1 += (double)pair_sum<V>(dv);
                s2 += (double)pair_sum<V>(d2);
                sd += (double)pair_sum<V>(da);
            }
            mean = fma(s1, 1.0 / NT, (double)c);
            m2 = fma(-s1, s1 * (1.0 / NT), s2);
            exact = s2 <= __DBL_MAX__ && !(sd > 0.0 && sd < 0x1p-60 * NT);
        }
        if (!exact) {
            double tot = 0.0;
#pragma unroll 1
            for (int k = 0; k < NL; ++k)
#pragma unroll 1
                for (int e = 0; e < V; ++e) tot += (double)load_one<GT>(t.g, pos(k, e));
            mean = tot * (1.0 / NT);
            m2 = 0.0;
#pragma unroll 1
            for (int k = 0; k < NL; ++k)
#pragma unroll 1
                for (int e = 0; e < V; ++e) {
                    const double dd = (double)load_one<GT>(t.g, pos(k, e)) - mean;
                    m2 = fma(dd, dd, m2);
                }
        }
#pragma unroll
        for (int off = 1, part = V * NL; off < 64; off <<= 1, part <<= 1) {
            const double om = __shfl_xor(mean, off, 64), om2 = __shfl_xor(m2, off, 64);
            sq += __shfl_xor(sq, off, 64);
            ab += __shfl_xor(ab, off, 64);
            merge_equal(mean, m2, om, om2, part);
        }
        const int w = threadIdx.x / 64;
        if ((threadIdx.x & 63) == 0) {
            lds4[w][0] = mean;
            lds4[w][1] = m2;
            lds4[w][2] = sq;
            lds4[w][3] = ab;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double mw[ST_WAVES], m2w[ST_WAVES];
            sq = ab = 0.0;
#pragma unroll
            for (int q = 0; q < ST_WAVES; ++q) {
                mw[q] = lds4[q][0];
                m2w[q] = lds4[q][1];
                sq += lds4[q][2];
                ab += lds4[q][3];
            }
#pragma unroll
            for (int h = 1; h < ST_WAVES; h <<= 1)
#pragma unroll
                for (int q = 0; q < ST_WAVES; q += 2 * h) merge_equal(mw[q], m2w[q], mw[q + h], m2w[q + h], 64 * V * NL * h);
            partials[4 * tile + 0] = mw[0] * (double)STAT_TILE;
            partials[4 * tile + 1] = m2w[0];
            partials[4 * tile + 2] = sq;
            partials[4 * tile + 3] = ab;
        }
        return;
    }
    const void *g = static_cast<const char *>(t.g) + base * (GT == GT_F32 ? 4 : 2);
    if constexpr (OFF16) {
        if (left >= STAT_TILE) {
            whole_f64<GT>(g, partials + 4 * tile, lds3, lds2);
            return;
        }
    }
    ragged_f64<GT>(g, (uint32_t)left, partials + 4 * tile, lds3, lds2);
}

// fp32 value of a sum of non-negative terms as an fp32 accumulator holds it:
// inf once the exact sum exceeds FLT_MAX.
__device__ __forceinline__ float f32_sum(double x) { return x > (double)__FLT_MAX__ ? __builtin_inff() : (float)x; }

__global__ __launch_bounds__(ST_THREADS) void stats_finish_kernel(const StatDesc *__restrict__ d,
                                                                  const double *__restrict__ partials,
                                                                  float *__restrict__ out)
{
    __shared__ double lds3[ST_WAVES][3];
    __shared__ double lds1[ST_WAVES][1];
    const StatDesc t = d[blockIdx.x];
    double s[3] = {0.0, 0.0, 0.0};      // sum g, sum g^2, sum |g|
    for (long long k = t.tile_begin + threadIdx.x; k < t.tile_end; k += ST_THREADS) {
        s[0] += partials[4 * k + 0];
        s[1] += partials[4 * k + 2];
        s[2] += partials[4 * k + 3];
    }
    block_sum<3>(s, lds3);
    const double N = (double)t.numel;
    const double mean = s[0] / N;
    // Chan et al.'s combination of the tiles' (count, mean, M2)
    double m2[1] = {0.0};
    for (long long k = t.tile_begin + threadIdx.x; k < t.tile_end; k += ST_THREADS) {
        const int64_t first = (k - t.tile_begin) * STAT_TILE;
        const double ni = (double)(t.numel - first < STAT_TILE ? t.numel - first : STAT_TILE);
        const double dm = partials[4 * k + 0] / ni - mean;
        m2[0] += fma(ni * dm, dm, partials[4 * k + 1]);
    }
    block_sum<1>(m2, lds1);
    if (threadIdx.x == 0) {
        // The reference's fp32 results: mean(g * g) and mean(|g|) from fp32 sums, std from
        // an fp32 M2 (torch's Welford accumulators on the GPU), then sqrt / divide / add in
        // fp32.  numel 0 gives NaN means and numel 0 or 1 a NaN std (unbiased), as torch does.
        const float sum_sq = f32_sum(s[1]), sum_abs = f32_sum(s[2]), m2f = f32_sum(m2[0]);
        const float mean_sq = sum_sq == __builtin_inff() ? sum_sq : (float)(s[1] / N);
        const float mean_abs = sum_abs == __builtin_inff() ? sum_abs : (float)(s[2] / N);
        const float sd = t.numel < 2 ? __builtin_nanf("")
                                     : (m2f == __builtin_inff() ? m2f : (float)sqrt(m2[0] / (N - 1.0)));
        out[3 * blockIdx.x + 0] = sqrtf(mean_sq);
        out[3 * blockIdx.x + 1] = sd / (mean_abs + 1e-12f);
        out[3 * blockIdx.x + 2] = mean_sq;
    }
}

// The scores of the bit decision (stquant_opt_simple.py:433-466): the EMAs with this
// decision's mean statistics folded in (the mean itself at the first decision), and per
// tensor 7.2 + log2(r_l / (r + 1e-12)) + log2(n_l / (n + 1e-12)) + log2(1 + 1 / cosh t)
// + log2(v_l / (v + 1e-12)), each operation rounded to fp32 in that order, so the bits are
// those of the same chain of torch operations (checked in tests/test_gpu_grad_stats.py).
// Bound by launches: as torch operations the chain is 24 of them, about 5 us of host time
// each.  A width-deciding optimizer step over GPT-2 small's 148 tensors 1776 -> 1387 us with
// this launch, once where the provisional scores settle no row, in place of the chain run twice.
__global__ __launch_bounds__(256) void scores_kernel(const float *__restrict__ stats, const float *__restrict__ mean,
                                                     int n, const float *__restrict__ t, float t_all,
                                                     const float *__restrict__ n_ema, const float *__restrict__ r_ema,
                                                     const float *__restrict__ v_ema, float a, float b,
                                                     float *__restrict__ out, float *__restrict__ ema)
{
    const float en = n_ema ? a * mean[0] + b * *n_ema : mean[0];
    const float er = n_ema ? a * mean[1] + b * *r_ema : mean[1];
    const float ev = n_ema ? a * mean[2] + b * *v_ema : mean[2];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) {
        ema[0] = en;
        ema[1] = er;
        ema[2] = ev;
    }
    if (i >= n) return;
    const float n_l = stats[3 * i], r_l = stats[3 * i + 1], v_l = stats[3 * i + 2];
    const float s_t = 1.0f + 1.0f / coshf(t ? t[i] : t_all);
    float s = 7.2f + log2f(r_l / (er + 1e-12f));
    s = s + log2f(n_l / (en + 1e-12f));
    s = s + log2f(s_t);
    s = s + log2f(v_l / (ev + 1e-12f));
    out[i] = s;
    out[n + i] = r_l;
}

}  // namespace

hipError_t launch_scores(const float *stats, const float *mean, int n, const float *t, float t_all, const float *n_ema,
                         const float *r_ema, const float *v_ema, float a, float b, float *out, float *ema, hipStream_t s)
{
    // without tensors one workgroup still writes the EMAs
    scores_kernel<<<dim3((unsigned)(n > 0 ? (n + 255) / 256 : 1)), dim3(256), 0, s>>>(stats, mean, n, t, t_all, n_ema, r_ema, v_ema,
                                                                         a, b, out, ema);
    return hipGetLastError();
}

hipError_t launch_grad_stats(const StatDesc *d, const long long *tb, int n, long long tiles, int grad_dt, bool off16,
                             double *partials, float *out, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (tiles > 0) {
        const auto partial = [&](auto kernel) {
            kernel<<<dim3((unsigned)tiles), dim3(ST_THREADS), 0, s>>>(d, n, tb, partials);
        };
        switch (grad_dt) {
        case GT_F32: partial(off16 ? stats_partial_kernel<GT_F32, true> : stats_partial_kernel<GT_F32, false>); break;
        case GT_BF16: partial(off16 ? stats_partial_kernel<GT_BF16, true> : stats_partial_kernel<GT_BF16, false>); break;
        default: partial(off16 ? stats_partial_kernel<GT_F16, true> : stats_partial_kernel<GT_F16, false>); break;
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    stats_finish_kernel<<<dim3((unsigned)n), dim3(ST_THREADS), 0, s>>>(d, partials, out);
    return hipGetLastError();
}

}  // namespace mdq
