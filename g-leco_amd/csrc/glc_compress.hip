// glc_compress.hip -- compress-side gfx950 kernels of libglc.
//
//   k_fit_*       per-partition overflow check + FP64 linear fit + max |delta|
//                 -> bit width (compression/CompressionKernels.cuh:46-218)
//   k_scan        exclusive scan of len*bits -> bit offsets
//                 (replaces the O(P^2) setBitOffsetsKernel, :222-238)
//   k_build_index 32-byte decode descriptors + 1024-element tile index
//   k_pack_*      bit packer: one wave per 1024-element tile, every word of the
//                 payload stored once, partial words merged inside a workgroup
//                 (replaces the per-element atomicOr packer, :243-372)
//   k_v6_*        GPUVariableLengthPartitionerV6 (compression/GpuPartitioner.cuh:34-214,
//                 compression/PartitioningKernels.cuh:648-744) without atomics
//                 or sorts: variance per block, radix selection of the three
//                 quartiles, counted prefix sum to emit partitions in order.
#include <hip/hip_runtime.h>

#include "glc_device.hpp"
#include "glc_internal.hpp"

namespace glc {
namespace {


// ---------------------------------------------------------------------------
// Fit.  The reference's block of `bs` threads (a multiple of 32, at most 256)
// sums over i = t, t + bs, ... in increasing i and reduces by the tree s = bs/2,
// bs/4, ..., 1 (:113-137); theta0/theta1 are bit-identical for the same
// contraction form when every value meets the same additions.  Three forms keep
// that order: a wave with the partition in registers (fit_wave_reg), a workgroup
// with it in registers (fit_block_reg), both reading it once, and a workgroup
// reading it twice (fit_block).  A fourth takes the other block sizes
// (fit_wave_any).
// ---------------------------------------------------------------------------

// Contraction form of the fit's FP64 expressions (:113-158 write a*b + c; the
// reference build lets nvcc fuse them, which the source does not show):
//   FORM 0: sum_xx += x*x and sum_xy += x*y as fma(x, x, s) / fma(x, y, s),
//           det = fma(n, Sxx, -(Sx*Sx)), num = fma(n, Sxy, -(Sx*Sy)),
//           theta0 = fma(-theta1, Sx, Sy) / n            (the default)
//   FORM 1: every product rounded on its own, no fma.
// The prediction fma(theta1, i, theta0) is the same in both forms.
template <int FORM> __device__ __forceinline__ double acc_prod(double a, double b, double s) {
    if constexpr (FORM == 0) return __builtin_fma(a, b, s);
    else return s + a * b;
}

// Sx = sum of i and Sxx = sum of i^2 over i < n without adding them up: where
// the tree takes in every thread (bs a power of two), each partial sum is an
// integer, below 2^53 for n <= kExactN, so every addition and product is exact
// in either form and in any order.
constexpr int32_t kExactN = 1 << 17;
__device__ __forceinline__ void exact_x_sums(int32_t n, double& Sx, double& Sxx) {
    const int64_t m = n;
    Sx = static_cast<double>(m * (m - 1) / 2);
    Sxx = static_cast<double>((m - 1) * m * (2 * m - 1) / 6);  // < 2^53 before the division
}

// theta from the four sums (:140-160): determinant test, then slope and
// intercept.
template <int FORM>
__device__ __forceinline__ void fit_theta(int32_t n, double Sx, double Sy, double Sxx, double Sxy, double& t0,
                                          double& t1) {
    const double dn = static_cast<double>(n);
    const double det = (FORM == 0) ? __builtin_fma(dn, Sxx, -(Sx * Sx)) : dn * Sxx - Sx * Sx;
    if (__builtin_fabs(det) > 1e-10) {
        t1 = ((FORM == 0) ? __builtin_fma(dn, Sxy, -(Sx * Sy)) : dn * Sxy - Sx * Sy) / det;
        t0 = ((FORM == 0) ? __builtin_fma(-t1, Sx, Sy) : Sy - t1 * Sx) / dn;
    } else {
        t1 = 0.0;
        t0 = Sy / dn;
    }
}

template <class T> __device__ __forceinline__ int64_t abs_delta(T val, double t0, double t1, int32_t i) {
    const int64_t dl = calc_delta<T>(val, enc_pred<T>(t0, t1, i));
    // -LLONG_MIN stays negative and is ignored by the max, as in :171-174
    return dl < 0 ? static_cast<int64_t>(0ULL - static_cast<uint64_t>(dl)) : dl;
}

template <class T, int TIER> __device__ __forceinline__ int64_t abs_delta_fast(T val, double t0, double t1, int32_t i) {
    const int64_t dl = enc_delta_fast<T, TIER>(val, t0, t1, i);
    return dl < 0 ? static_cast<int64_t>(0ULL - static_cast<uint64_t>(dl)) : dl;
}

// enc_tier of a partition's n predictions
template <class T> __device__ __forceinline__ int fit_tier(int32_t n, double t0, double t1) {
    return enc_tier<T>(__builtin_fma(t1, 0.0, t0), __builtin_fma(t1, static_cast<double>(n - 1), t0));
}

__device__ __forceinline__ int32_t bits_for(int64_t m) {
    if (m <= 0) return 0;
    const int32_t bb = 64 - __builtin_clzll(static_cast<unsigned long long>(m)) + 1;
    return bb > 64 ? 64 : bb;
}

// The fit's outputs, one entry per partition.
struct FitOut {
    int32_t* __restrict__ type;
    double* __restrict__ params;
    int32_t* __restrict__ bits;
    int64_t* __restrict__ err;
};
// one thread
__device__ __forceinline__ void fit_store(const FitOut& o, int64_t p, double t0, double t1, int64_t mx) {
    o.type[p] = MODEL_LINEAR;
    o.params[4 * p] = t0; o.params[4 * p + 1] = t1; o.params[4 * p + 2] = 0.0; o.params[4 * p + 3] = 0.0;
    o.err[p] = mx;
    o.bits[p] = bits_for(mx);
}
template <class T> __device__ __forceinline__ void fit_store_direct(const FitOut& o, int64_t p) {  // :95-106 DIRECT_COPY
    o.type[p] = MODEL_DIRECT_COPY;
    o.params[4 * p] = 0.0; o.params[4 * p + 1] = 0.0; o.params[4 * p + 2] = 0.0; o.params[4 * p + 3] = 0.0;
    o.err[p] = 0;
    o.bits[p] = static_cast<int32_t>(sizeof(T) * 8);
}

__device__ __forceinline__ int64_t wave_max_i64(int64_t mx) {
    for (int o = 32; o > 0; o >>= 1) {
        const int64_t y = __shfl_xor(mx, o, 64);
        mx = y > mx ? y : mx;
    }
    return mx;
}

// A zero the compiler cannot see through.  Index values that depend only on
// the lane (i, (double)i, i*i) are loop invariants of a loop over
// partitions; hoisted out of it they would stay live in registers for the
// whole loop, and the max-error pass would keep the sums pass's (double)i
// of every value.
__device__ __forceinline__ int32_t opaque_zero() {
    int32_t z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return z;
}

// Block size 256, partition p of 0 < n <= 512 * NSTEP values, by one wave that
// holds it in registers: lane l plays the reference's threads l, l+64, l+128 and
// l+192 (sets j = 0..3), value i = 64 j + l in set j & 3, increasing i within a
// set.  The tree's steps 128 and 64 add sets inside a lane (sum[t] += sum[t + s]
// with t + s in set j + s/64 of the same lane), 32..1 are shuffles; the max-error
// pass reads the same registers.  No LDS, no barrier.
constexpr int kFitWaves = 4;
constexpr int kFitWaveBs = 256;

// Both register forms work in FP64 throughout.  64-bit values are kept as the
// doubles that the sums need anyway (32-bit ones as they are): with |y| <= 2^52
// and predictions of tier 1, |y - round(pr)| is the difference of two integers
// below 2^53 in magnitude, exact, and equals |calc_delta|.  FULL: every lane
// has a value in every row; else a lane past n sums 0 (x + 0 = x, and no sum is
// ever -0) and adds no residual.  16 instead of 45 vector instructions a value for
// int64: instructions were 2/3 of the time.  Values above 2^52, tier 2 and
// predictions that may saturate read the partition again (fit_again).
constexpr double kFitExact = 4503599627370496.0;  // 2^52
template <class T> using FitKeep = typename std::conditional<sizeof(T) == 8, double, T>::type;

// Largest residual of values i = i0, i0 + step, ... < n, read from memory, in
// integers; -1: a uint64 above 2^53 (DIRECT_COPY).  One lane's share.
template <class T>
__device__ __forceinline__ int64_t fit_again(const T* __restrict__ x, int32_t i0, int32_t n, int32_t step, double t0,
                                             double t1) {
    const int tier = fit_tier<T>(n, t0, t1);
    int64_t mx = 0;
    int ovf = 0;
    for (int32_t base = i0; base < n; base += 8 * step) {
        T y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int32_t i = base + k * step;
            y[k] = x[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // the clamped index repeats element n - 1: same value
            const int32_t i = base + k * step, j = i < n ? i : n - 1;
            ovf |= might_overflow_double<T>(y[k]) ? 1 : 0;
            int64_t ab;
            if (tier == 1) ab = abs_delta_fast<T, 1>(y[k], t0, t1, j);
            else if (std::is_same<T, int64_t>::value && tier == 2) ab = abs_delta_fast<T, 2>(y[k], t0, t1, j);
            else ab = abs_delta<T>(y[k], t0, t1, j);
            mx = ab > mx ? ab : mx;
        }
    }
    return ovf ? -1 : mx;
}

// |y - round(pr)| of value i
template <class K> __device__ __forceinline__ double fit_resid(K y, double xi, double t0, double t1) {
    return __builtin_fabs(static_cast<double>(y) - round_away(__builtin_fma(t1, xi, t0)));
}

template <class T, int FORM, int NSTEP, bool FULL>
__device__ __forceinline__ void fit_wave_form(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o,
                                              int lane_) {
    constexpr int J = 8 * NSTEP;
    const int lane = lane_ + opaque_zero();
    T raw[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {  // branch-free: every load in flight at once
        const int32_t i = 64 * j + lane;
        raw[j] = x[FULL || i < n ? i : n - 1];
    }
    FitKeep<T> y[J];
    double b[4] = {0.0, 0.0, 0.0, 0.0}, d[4] = {0.0, 0.0, 0.0, 0.0}, top = 0.0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int32_t i = 64 * j + lane;
        y[j] = FULL || i < n ? static_cast<FitKeep<T>>(raw[j]) : FitKeep<T>(0);
        const double yi = static_cast<double>(y[j]);
        b[j & 3] = b[j & 3] + yi;
        d[j & 3] = acc_prod<FORM>(static_cast<double>(i), yi, d[j & 3]);
        if constexpr (sizeof(T) == 8) top = __builtin_fmax(top, __builtin_fabs(yi));
    }
    double Sy = (b[0] + b[2]) + (b[1] + b[3]);
    double Sxy = (d[0] + d[2]) + (d[1] + d[3]);
    for (int h = 32; h > 0; h >>= 1) {
        Sy = Sy + __shfl_down(Sy, h, 64);
        Sxy = Sxy + __shfl_down(Sxy, h, 64);
    }
    // lane 0 holds the sums; every lane computes the same theta from them
    Sy = __shfl(Sy, 0, 64);
    Sxy = __shfl(Sxy, 0, 64);
    double Sx, Sxx, t0, t1;
    exact_x_sums(n, Sx, Sxx);
    fit_theta<FORM>(n, Sx, Sy, Sxx, Sxy, t0, t1);
    const int lane2 = lane_ + opaque_zero();  // (double)i afresh: not kept live from the sums pass
    const bool exact = sizeof(T) == 4 || !__any(!(top <= kFitExact));
    int64_t mx;
    if (exact && fit_tier<T>(n, t0, t1) == 1) {
        double md = 0.0;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int32_t i = 64 * j + lane2;
            const double r = fit_resid(y[j], static_cast<double>(i), t0, t1);
            md = __builtin_fmax(md, FULL || i < n ? r : 0.0);
        }
        mx = static_cast<int64_t>(md);
    } else {
        mx = fit_again<T>(x, lane2, n, 64, t0, t1);
        if (__any(mx < 0 && !std::is_signed<T>::value)) {
            if (lane == 0) fit_store_direct<T>(o, p);
            return;
        }
    }
    mx = wave_max_i64(mx);
    if (lane == 0) fit_store(o, p, t0, t1, mx);
}

template <class T, int FORM, int NSTEP>
__device__ __forceinline__ void fit_wave_reg(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o, int lane) {
    if (n == 512 * NSTEP) fit_wave_form<T, FORM, NSTEP, true>(x, n, p, o, lane);
    else fit_wave_form<T, FORM, NSTEP, false>(x, n, p, o, lane);
}

// Any block size, any n, by one wave: lane l plays threads l + 64 j < bs, the
// tree runs through s_t (bs doubles), truncated as the reference's is for block
// sizes that are no power of two.  The block size is 256 except where the
// column's first partition has at most 224 values, which for fixed sizes means
// that all are as short: two values a thread at most.
template <class T, int FORM>
__device__ __forceinline__ void fit_wave_any(const T* __restrict__ x, int32_t n, int bs, int64_t p, const FitOut& o,
                                             int lane, double* __restrict__ s_t) {
    double s[4][4] = {};  // sums x, y, xx, xy of sets j = 0..3
    int ovf = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = lane + 64 * j;
        if (t < bs) {
            for (int32_t i = t; i < n; i += bs) {
                const T val = x[i];
                ovf |= might_overflow_double<T>(val) ? 1 : 0;
                const double xi = static_cast<double>(i), yi = static_cast<double>(val);
                s[0][j] = s[0][j] + xi;
                s[1][j] = s[1][j] + yi;
                s[2][j] = acc_prod<FORM>(xi, xi, s[2][j]);
                s[3][j] = acc_prod<FORM>(xi, yi, s[3][j]);
            }
        }
    }
    if (__any(ovf)) {
        if (lane == 0) fit_store_direct<T>(o, p);
        return;
    }
    double tot[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < bs) s_t[lane + 64 * j] = s[q][j];
        wave_lds_fence();
        for (int h = bs >> 1; h > 0; h >>= 1) {  // reads [h, 2h), writes [0, h)
            for (int t = lane; t < h; t += 64) s_t[t] = s_t[t] + s_t[t + h];
            wave_lds_fence();
        }
        tot[q] = s_t[0];
        wave_lds_fence();  // s_t is the next sum's
    }
    double t0, t1;
    fit_theta<FORM>(n, tot[0], tot[1], tot[2], tot[3], t0, t1);
    int64_t mx = 0;
    for (int32_t i = lane; i < n; i += 64) {
        const int64_t ab = abs_delta<T>(x[i], t0, t1, i);
        mx = ab > mx ? ab : mx;
    }
    mx = wave_max_i64(mx);
    if (lane == 0) fit_store(o, p, t0, t1, mx);
}

// Any block size, any n > 0, by a 256-thread workgroup: threads t < bs sum
// with eight loads in flight, the tree runs through s_t, all threads take the
// maximum.  Uniform arguments.
template <class T, int FORM>
__device__ __forceinline__ void fit_block_any(const T* __restrict__ x, int32_t n, int bs, int64_t p, const FitOut& o,
                                              double* __restrict__ s_t, int64_t* __restrict__ s_mx) {
    constexpr int K = 8;
    const int tid = threadIdx.x;
    const uint32_t un = static_cast<uint32_t>(n);  // indices past n may pass 2^31
    double s[4] = {};  // sums x, y, xx, xy
    int ovf = 0;
    if (tid < bs) {
        for (uint32_t base = tid; base < un; base += bs * K) {
            T y[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t i = base + bs * k;
                y[k] = x[i < un ? i : un - 1];
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const uint32_t i = base + bs * k;
                if (i < un) {
                    ovf |= might_overflow_double<T>(y[k]) ? 1 : 0;
                    const double xi = static_cast<double>(i), yi = static_cast<double>(y[k]);
                    s[0] = s[0] + xi;
                    s[1] = s[1] + yi;
                    s[2] = acc_prod<FORM>(xi, xi, s[2]);
                    s[3] = acc_prod<FORM>(xi, yi, s[3]);
                }
            }
        }
    }
    if (__syncthreads_or(ovf)) {
        if (tid == 0) fit_store_direct<T>(o, p);
        return;
    }
    double tot[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (tid < bs) s_t[tid] = s[q];
        __syncthreads();
        for (int h = bs >> 1; h > 0; h >>= 1) {
            if (tid < h) s_t[tid] = s_t[tid] + s_t[tid + h];
            __syncthreads();
        }
        tot[q] = s_t[0];
        __syncthreads();
    }
    double t0, t1;
    fit_theta<FORM>(n, tot[0], tot[1], tot[2], tot[3], t0, t1);
    int64_t mx = 0;
    const bool fast = fit_tier<T>(n, t0, t1) == 1;
    for (uint32_t base = tid; base < un; base += 256 * K) {
        T y[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t i = base + 256 * k;
            y[k] = x[i < un ? i : un - 1];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {  // the clamped index repeats element n - 1: same value
            const uint32_t i = base + 256 * k;
            const int32_t j = static_cast<int32_t>(i < un ? i : un - 1);
            const int64_t ab = fast ? abs_delta_fast<T, 1>(y[k], t0, t1, j) : abs_delta<T>(y[k], t0, t1, j);
            mx = ab > mx ? ab : mx;
        }
    }
    mx = wave_max_i64(mx);
    if ((tid & 63) == 0) s_mx[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 4; ++w) mx = s_mx[w] > mx ? s_mx[w] : mx;
        fit_store(o, p, t0, t1, mx);
    }
    __syncthreads();  // s_t and s_mx are the next partition's
}

// The reference's block itself (256 threads): the tree of NS sums per thread,
// s = 128 and 64 through LDS, 32..1 by shuffles in wave 0; theta to every thread.
struct FitLds {
    double sum[4][128];
    double th[2];
    int64_t mx[4];
};

template <int NS> __device__ __forceinline__ void block_tree(double (&s)[NS], FitLds& L) {  // result in thread 0
    const int tid = threadIdx.x;
    if (tid >= 128)
#pragma unroll
        for (int q = 0; q < NS; ++q) L.sum[q][tid - 128] = s[q];
    __syncthreads();
    if (tid < 128)
#pragma unroll
        for (int q = 0; q < NS; ++q) s[q] = s[q] + L.sum[q][tid];
    __syncthreads();
    if (tid >= 64 && tid < 128)
#pragma unroll
        for (int q = 0; q < NS; ++q) L.sum[q][tid - 64] = s[q];
    __syncthreads();
    if (tid < 64) {
#pragma unroll
        for (int q = 0; q < NS; ++q) s[q] = s[q] + L.sum[q][tid];
        for (int h = 32; h > 0; h >>= 1)
#pragma unroll
            for (int q = 0; q < NS; ++q) s[q] = s[q] + __shfl_down(s[q], h, 64);
    }
}

__device__ __forceinline__ void block_store(const FitOut& o, int64_t p, double t0, double t1, int64_t mx, FitLds& L) {
    mx = wave_max_i64(mx);
    if ((threadIdx.x & 63) == 0) L.mx[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t m = L.mx[0];
        for (int w = 1; w < 4; ++w) m = L.mx[w] > m ? L.mx[w] : m;
        fit_store(o, p, t0, t1, m);
    }
    __syncthreads();  // L is the workgroup's next partition's
}

// Block size 256, 0 < n <= 256 K values, by a workgroup: thread t holds its
// values i = t, t+256, ... in registers for both passes.  Uniform arguments.
template <class T, int FORM, int K, bool FULL>
__device__ __forceinline__ void fit_block_form(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o,
                                               FitLds& L) {
    const int tid = static_cast<int>(threadIdx.x) + opaque_zero();
    T raw[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {  // branch-free: every load in flight at once
        const int32_t i = tid + 256 * k;
        raw[k] = x[FULL || i < n ? i : n - 1];
    }
    FitKeep<T> y[K];
    double s[2] = {0.0, 0.0}, top = 0.0;  // sums y, xy
#pragma unroll
    for (int k = 0; k < K; ++k) {  // CompressionKernels.cuh:113-120, thread t's own order
        const int32_t i = tid + 256 * k;
        y[k] = FULL || i < n ? static_cast<FitKeep<T>>(raw[k]) : FitKeep<T>(0);
        const double yi = static_cast<double>(y[k]);
        s[0] = s[0] + yi;
        s[1] = acc_prod<FORM>(static_cast<double>(i), yi, s[1]);
        if constexpr (sizeof(T) == 8) top = __builtin_fmax(top, __builtin_fabs(yi));
    }
    const bool exact = sizeof(T) == 4 || !__syncthreads_or(!(top <= kFitExact));
    block_tree<2>(s, L);
    if (tid == 0) {
        double Sx, Sxx;
        exact_x_sums(n, Sx, Sxx);
        fit_theta<FORM>(n, Sx, s[0], Sxx, s[1], L.th[0], L.th[1]);
    }
    __syncthreads();
    const double t0 = L.th[0], t1 = L.th[1];
    const int tid2 = static_cast<int>(threadIdx.x) + opaque_zero();  // (double)i afresh, as in fit_wave_reg
    int64_t mx;
    if (exact && fit_tier<T>(n, t0, t1) == 1) {
        double md = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int32_t i = 256 * k + tid2;
            const double r = fit_resid(y[k], static_cast<double>(i), t0, t1);
            md = __builtin_fmax(md, FULL || i < n ? r : 0.0);
        }
        mx = static_cast<int64_t>(md);
    } else {
        mx = fit_again<T>(x, tid2, n, 256, t0, t1);
        if (!std::is_signed<T>::value && __syncthreads_or(mx < 0)) {
            if (tid == 0) fit_store_direct<T>(o, p);
            return;
        }
    }
    block_store(o, p, t0, t1, mx, L);
}

template <class T, int FORM, int K>
__device__ __forceinline__ void fit_block_reg(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o,
                                              FitLds& L) {
    if (n == 256 * K) fit_block_form<T, FORM, K, true>(x, n, p, o, L);
    else fit_block_form<T, FORM, K, false>(x, n, p, o, L);
}

// Block size 256, any n > 0, by a workgroup that reads the partition twice:
// eight loads a thread in flight; the max-error pass goes from the end back (the
// part read last is the one most likely still cached; a maximum has no order).
template <class T, int FORM>
__device__ __forceinline__ void fit_block(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o, FitLds& L) {
    constexpr int K = 8, kStep = 256 * K;
    const int tid = threadIdx.x;
    double s[4] = {0.0, 0.0, 0.0, 0.0};  // sums y, xy, x, xx
    int ovf = 0;
    const bool xs = n > kExactN;
    for (uint32_t step = 0; step < static_cast<uint32_t>(n); step += kStep) {  // passes 2^31 at the largest n
        const int32_t base = static_cast<int32_t>(step);
        T y[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int32_t i = base + tid + 256 * k;
            y[k] = x[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int32_t i = base + tid + 256 * k;
            if (i < n) {
                ovf |= might_overflow_double<T>(y[k]) ? 1 : 0;
                const double xi = static_cast<double>(i), yi = static_cast<double>(y[k]);
                s[0] = s[0] + yi;
                s[1] = acc_prod<FORM>(xi, yi, s[1]);
                if (xs) {
                    s[2] = s[2] + xi;
                    s[3] = acc_prod<FORM>(xi, xi, s[3]);
                }
            }
        }
    }
    if (__syncthreads_or(ovf)) {
        if (tid == 0) fit_store_direct<T>(o, p);
        return;
    }
    block_tree<4>(s, L);
    if (tid == 0) {
        double Sx = s[2], Sxx = s[3];
        if (!xs) exact_x_sums(n, Sx, Sxx);
        fit_theta<FORM>(n, Sx, s[0], Sxx, s[1], L.th[0], L.th[1]);
    }
    __syncthreads();
    const double t0 = L.th[0], t1 = L.th[1];
    int64_t mx = 0;
    const bool fast = fit_tier<T>(n, t0, t1) == 1;
    for (int32_t base = (n - 1) / kStep * kStep; base >= 0; base -= kStep) {
        T y[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int32_t i = base + tid + 256 * k;
            y[k] = x[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {  // the clamped index repeats element n - 1: same value
            const int32_t i = base + tid + 256 * k, j = i < n ? i : n - 1;
            const int64_t ab = fast ? abs_delta_fast<T, 1>(y[k], t0, t1, j) : abs_delta<T>(y[k], t0, t1, j);
            mx = ab > mx ? ab : mx;
        }
    }
    block_store(o, p, t0, t1, mx, L);
}

// Sizes of the forms (block size 256).  A wave holds up to 2048 values, a
// workgroup 8192; above, two reads.
constexpr int32_t kFitWaveMax = 2048;
constexpr int32_t kFitRegMax = 8192;

// Fixed partitions of at most S values, S <= 512 * NSTEP: a wave each.
template <class T, int FORM, int NSTEP>
__global__ __launch_bounds__(64 * kFitWaves) void k_fit_waves(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                              const int32_t* __restrict__ en, FitOut o, int64_t P) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * kFitWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (p >= P) return;
    const int32_t s0 = st[p];
    const int32_t n = en[p] - s0;
    if (n > 0) fit_wave_reg<T, FORM, NSTEP>(v + s0, n, p, o, threadIdx.x & 63);
}

// Fixed partitions of at most S values, S <= 256 K (K = 0: any): a workgroup each.
template <class T, int FORM, int K>
__global__ __launch_bounds__(256) void k_fit_block(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                   const int32_t* __restrict__ en, FitOut o, int64_t P) {
    __shared__ FitLds L;
    const int64_t p = blockIdx.x;
    const int32_t s0 = st[p];
    const int32_t n = en[p] - s0;
    if (n <= 0) return;
    if constexpr (K > 0) fit_block_reg<T, FORM, K>(v + s0, n, p, o, L);
    else fit_block<T, FORM>(v + s0, n, p, o, L);
}

// Mixed sizes (V6, split/merge, explicit partitions), block size 256: workgroup
// g takes partitions g * chunk .. + chunk.  Its waves first fit the partitions of
// at most kFitWaveMax values, one each, round robin; then the whole workgroup
// fits the longer ones, one after the other.  Results do not depend on who fits a
// partition.  chunk: 16 for long lists (2^28 uint64 V6, 122880 partitions: chunks of
// 4 / 16 / 64 took 492 / 484 / 497 us), down to 1 where workgroups would be too few
// (3500 partitions of 20000 values, split/merge 2^26: 618 -> 186 us).
// MINW: waves a SIMD.  With four the 64-bit forms are short of 2 to 10 registers
// and spill, which the forms that hold 32 values a lane pay for most (2^28 uint64
// V6 base 2048: 413 us with four, 389 with three; 2^27 int64 base 4096: 234, 214);
// short partitions and ones of many passes want the fourth wave (2^27 uint64 base
// 512: 355, 365; split/merge 2^26: 186, 193).
template <class T, int FORM, int MINW>
__global__ __launch_bounds__(256, MINW) void k_fit_chunk(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                   const int32_t* __restrict__ en, FitOut o, int64_t P, int chunk) {
    __shared__ FitLds L;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * chunk;
    const int64_t p1 = (p0 + chunk < P) ? p0 + chunk : P;
    for (int64_t p = p0 + wave; p < p1; p += 4) {
        const int32_t s0 = st[p];
        const int32_t n = en[p] - s0;
        if (n <= 0) continue;  // :62, entry keeps its initial values
        if (n <= 1024) fit_wave_reg<T, FORM, 2>(v + s0, n, p, o, lane);
        else if (n <= kFitWaveMax) fit_wave_reg<T, FORM, 4>(v + s0, n, p, o, lane);
    }
    for (int64_t p = p0; p < p1; ++p) {  // uniform over the workgroup
        const int32_t s0 = st[p];
        const int32_t n = en[p] - s0;
        if (n <= kFitWaveMax) continue;
        if (n <= kFitRegMax / 2) fit_block_reg<T, FORM, 16>(v + s0, n, p, o, L);
        else if (n <= kFitRegMax) fit_block_reg<T, FORM, 32>(v + s0, n, p, o, L);
        else fit_block<T, FORM>(v + s0, n, p, o, L);
    }
}

// Other block sizes, in chunks as k_fit_chunk: partitions of up to 1024 values
// a wave each, longer ones (mixed sizes whose first partition is short) the
// workgroup.  2e7 int64 values in partitions of 64: 263 us where a workgroup per
// partition took 602.
constexpr int kFitAnyMax = 224;  // the largest block size below 256
template <class T, int FORM>
__global__ __launch_bounds__(64 * kFitWaves) void k_fit_any(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                            const int32_t* __restrict__ en, FitOut o, int64_t P,
                                                            int bs, int chunk) {
    __shared__ double s_t[kFitWaves][kFitAnyMax];
    __shared__ int64_t s_mx[kFitWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * chunk;
    const int64_t p1 = (p0 + chunk < P) ? p0 + chunk : P;
    int longer = 0;
    for (int64_t p = p0 + wave; p < p1; p += kFitWaves) {
        const int32_t s0 = st[p];
        const int32_t n = en[p] - s0;
        if (n > 1024) longer = 1;
        else if (n > 0) fit_wave_any<T, FORM>(v + s0, n, bs, p, o, threadIdx.x & 63, s_t[wave]);
    }
    if (!__syncthreads_or(longer)) return;
    for (int64_t p = p0; p < p1; ++p) {
        const int32_t s0 = st[p];
        const int32_t n = en[p] - s0;
        if (n > 1024) fit_block_any<T, FORM>(v + s0, n, bs, p, o, s_t[0], s_mx);
    }
}

// Block size 256, any n > 0, by one wave reading the partition twice (batches
// with partitions above kFitWaveMax): fit_wave_reg's order, 512 values a step,
// eight loads in flight.
template <class T, int FORM>
__device__ __forceinline__ void fit_wave_long(const T* __restrict__ x, int32_t n, int64_t p, const FitOut& o,
                                              int lane) {
    double a[4] = {}, b[4] = {}, c[4] = {}, d[4] = {};
    int ovf = 0;
    const bool xs = n > kExactN;
    for (uint32_t step = 0; step < static_cast<uint32_t>(n); step += 2 * kFitWaveBs) {  // passes 2^31 at the largest n
        const int32_t base = static_cast<int32_t>(step);
        T y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int32_t i = base + 64 * k + lane;
            y[k] = x[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int32_t i = base + 64 * k + lane;
            if (i < n) {
                ovf |= might_overflow_double<T>(y[k]) ? 1 : 0;
                const double xi = static_cast<double>(i), yi = static_cast<double>(y[k]);
                b[k & 3] = b[k & 3] + yi;
                d[k & 3] = acc_prod<FORM>(xi, yi, d[k & 3]);
                if (xs) {
                    a[k & 3] = a[k & 3] + xi;
                    c[k & 3] = acc_prod<FORM>(xi, xi, c[k & 3]);
                }
            }
        }
    }
    if (__any(ovf)) {
        if (lane == 0) fit_store_direct<T>(o, p);
        return;
    }
    double s[4] = {(b[0] + b[2]) + (b[1] + b[3]), (d[0] + d[2]) + (d[1] + d[3]), (a[0] + a[2]) + (a[1] + a[3]),
                   (c[0] + c[2]) + (c[1] + c[3])};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        for (int h = 32; h > 0; h >>= 1) s[q] = s[q] + __shfl_down(s[q], h, 64);
        s[q] = __shfl(s[q], 0, 64);
    }
    if (!xs) exact_x_sums(n, s[2], s[3]);
    double t0, t1;
    fit_theta<FORM>(n, s[2], s[0], s[3], s[1], t0, t1);
    int64_t mx = 0;
    const bool fast = fit_tier<T>(n, t0, t1) == 1;
    for (int32_t base = (n - 1) / (2 * kFitWaveBs) * (2 * kFitWaveBs); base >= 0; base -= 2 * kFitWaveBs) {
        T y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int32_t i = base + 64 * k + lane;
            y[k] = x[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // the clamped index repeats element n - 1: same value
            const int32_t i = base + 64 * k + lane, j = i < n ? i : n - 1;
            const int64_t ab = fast ? abs_delta_fast<T, 1>(y[k], t0, t1, j) : abs_delta<T>(y[k], t0, t1, j);
            mx = ab > mx ? ab : mx;
        }
    }
    mx = wave_max_i64(mx);
    if (lane == 0) fit_store(o, p, t0, t1, mx);
}

// Batched fit, a wave per partition, every element type in one launch (the
// type comes from the column).  NMAX: the longest partition of the batch, 1024
// (92 VGPRs instead of 124, five waves a SIMD; held to seven waves it spills 84
// bytes: 1000 columns, 2^26 values 100 against 91 us), 2048, or 0 for longer ones,
// which take two reads in the wave.
template <class T, int NMAX>
__device__ __forceinline__ void fit_batch_one(const BatchCol& c, int64_t p, int32_t s0, int32_t n, int lane,
                                              double* s_t) {
    const FitOut o{c.type, c.params, c.bits, c.err};
    const T* x = static_cast<const T*>(c.values) + s0;
    if (c.fit_bs != kFitWaveBs) fit_wave_any<T, 0>(x, n, c.fit_bs, p, o, lane, s_t);
    else if (NMAX == 1024 || n <= 1024) fit_wave_reg<T, 0, 2>(x, n, p, o, lane);
    else if (NMAX == 2048 || n <= kFitWaveMax) fit_wave_reg<T, 0, NMAX == 1024 ? 2 : 4>(x, n, p, o, lane);
    else if constexpr (NMAX == 0) fit_wave_long<T, 0>(x, n, p, o, lane);
}

template <int NMAX>
__global__ __launch_bounds__(64 * kFitWaves, NMAX == 1024 ? 5 : 4) void k_fit_wave_batch(
    const BatchCol* __restrict__ cols, const int32_t* __restrict__ part_col, int64_t Ptot, int32_t S) {
    __shared__ double s_t[kFitWaves][kFitAnyMax];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t g = static_cast<int64_t>(blockIdx.x) * kFitWaves + wave;
    if (g >= Ptot) return;
    const BatchCol& c = cols[part_col[g]];
    const int64_t p = g - c.part_base;
    const int32_t s0 = static_cast<int32_t>(p * S);  // as k_fixed_parts_batch writes them; no load to wait for
    const int32_t n = static_cast<int32_t>(c.n - s0 < S ? c.n - s0 : S);
    if (n <= 0) return;
    switch (c.dtype) {
        case GLC_I32: fit_batch_one<int32_t, NMAX>(c, p, s0, n, lane, s_t[wave]); break;
        case GLC_U32: fit_batch_one<uint32_t, NMAX>(c, p, s0, n, lane, s_t[wave]); break;
        case GLC_I64: fit_batch_one<int64_t, NMAX>(c, p, s0, n, lane, s_t[wave]); break;
        default: fit_batch_one<uint64_t, NMAX>(c, p, s0, n, lane, s_t[wave]); break;
    }
}

// ---------------------------------------------------------------------------
// Single-workgroup exclusive scan of int64 values produced by a functor.
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 1024;

struct LenBits {
    const int32_t* st;
    const int32_t* en;
    const int32_t* bits;
    __device__ int64_t operator()(int64_t p) const {
        return static_cast<int64_t>(en[p] - st[p]) * static_cast<int64_t>(bits[p]);
    }
};

// Exclusive scan of f(0..P-1) into out[] and the sum into *total, in three
// launches of 1024-value tiles (all loads coalesced).  out[] doubles as the
// scratch for the tile sums: tile b's sum is parked in out[b * 1024] until
// the down-sweep overwrites it with the final value.
template <int NT = kScanThreads>
__device__ __forceinline__ int64_t block_excl_scan(int64_t x, int64_t* s_w, int64_t* total) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int64_t v = x;
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t y = __shfl_up(v, o, 64);
        if (lane >= o) v += y;
    }
    if (lane == 63) s_w[w] = v;
    __syncthreads();
    if (tid == 0) {
        int64_t acc = 0;
        for (int k = 0; k < NT / 64; ++k) {
            const int64_t t = s_w[k];
            s_w[k] = acc;
            acc += t;
        }
        s_w[NT / 64] = acc;
    }
    __syncthreads();
    const int64_t r = s_w[w] + v - x;
    *total = s_w[NT / 64];
    __syncthreads();
    return r;
}

template <class F> __global__ __launch_bounds__(kScanThreads) void k_scan_up(F f, int64_t P, int64_t* __restrict__ out) {
    __shared__ int64_t s_w[kScanThreads / 64 + 1];
    const int64_t p = static_cast<int64_t>(blockIdx.x) * kScanThreads + threadIdx.x;
    int64_t tot;
    (void)block_excl_scan(p < P ? f(p) : 0, s_w, &tot);
    if (threadIdx.x == 0) out[static_cast<int64_t>(blockIdx.x) * kScanThreads] = tot;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_mid(int64_t* __restrict__ out, int64_t nb,
                                                           int64_t* __restrict__ total) {
    __shared__ int64_t s_w[kScanThreads / 64 + 1];
    int64_t carry = 0;
    for (int64_t b0 = 0; b0 < nb; b0 += kScanThreads) {
        const int64_t b = b0 + threadIdx.x;
        const int64_t x = b < nb ? out[b * kScanThreads] : 0;
        int64_t tot;
        const int64_t e = block_excl_scan(x, s_w, &tot);
        if (b < nb) out[b * kScanThreads] = carry + e;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

template <class F> __global__ __launch_bounds__(kScanThreads) void k_scan_down(F f, int64_t P, int64_t* __restrict__ out) {
    __shared__ int64_t s_w[kScanThreads / 64 + 1];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanThreads;
    const int64_t p = base + threadIdx.x;
    const int64_t carry = out[base];
    int64_t tot;
    const int64_t e = block_excl_scan(p < P ? f(p) : 0, s_w, &tot);  // all threads have read carry
    if (p < P) out[p] = carry + e;
}

template <class F> int launch_scan(F f, int64_t P, int64_t* out, int64_t* total, hipStream_t s) {
    if (P <= 0) return fail(GLC_ERR_STATE, "empty scan");
    const int64_t nb = (P + kScanThreads - 1) / kScanThreads;
    hipLaunchKernelGGL(k_scan_up<F>, dim3(static_cast<unsigned>(nb)), dim3(kScanThreads), 0, s, f, P, out);
    hipLaunchKernelGGL(k_scan_mid, dim3(1), dim3(kScanThreads), 0, s, out, nb, total);
    hipLaunchKernelGGL(k_scan_down<F>, dim3(static_cast<unsigned>(nb)), dim3(kScanThreads), 0, s, f, P, out);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

// Batched offsets: one workgroup per column scans that column's partitions
// and reserves the column's payload words in *col_words.
__global__ __launch_bounds__(kScanThreads) void k_scan_batch(const BatchCol* __restrict__ cols,
                                                             int64_t* __restrict__ col_bits) {
    const BatchCol& c = cols[blockIdx.x];
    LenBits f{c.start, c.end, c.bits};
    __shared__ int64_t s[kScanThreads];
    const int tid = threadIdx.x;
    const int64_t P = c.P;
    const int64_t chunk = (P + kScanThreads - 1) / kScanThreads;
    const int64_t b0 = tid * chunk;
    const int64_t b1 = (b0 + chunk < P) ? b0 + chunk : P;
    int64_t local = 0;
    for (int64_t p = b0; p < b1; ++p) local += f(p);
    s[tid] = local;
    __syncthreads();
    for (int o = 1; o < kScanThreads; o <<= 1) {
        int64_t y = (tid >= o) ? s[tid - o] : 0;
        __syncthreads();
        s[tid] += y;
        __syncthreads();
    }
    int64_t acc = s[tid] - local;
    for (int64_t p = b0; p < b1; ++p) {
        c.off[p] = acc;
        acc += f(p);
    }
    if (tid == kScanThreads - 1) col_bits[blockIdx.x] = s[tid];
}

// ---------------------------------------------------------------------------
// Decode index: Desc[P] + tile_part[] + validation summary.
// ---------------------------------------------------------------------------
// Wave-wide max of a value every lane holds (no lane has exited).
template <class V> __device__ __forceinline__ V wave_max_all(V x) {
    for (int o = 32; o > 0; o >>= 1) {
        const V y = __shfl_xor(x, o, 64);
        x = y > x ? y : x;
    }
    return x;
}

// One thread per partition, kIndexThreads per workgroup.  The column
// summary (flags, max bits, total bits) is reduced across each wave and then
// across the workgroup in LDS, so each workgroup issues one atomic per field:
// same-address device atomics serialize, and one set per wave cost ~50 us on
// 1.2e5 partitions.
constexpr int kIndexThreads = 1024;
struct IndexIn {
    const int32_t* __restrict__ st;
    const int32_t* __restrict__ en;
    const int32_t* __restrict__ type;
    const double* __restrict__ params;
    const int32_t* __restrict__ bits;
    int64_t P, n, n_index;
    Desc* __restrict__ desc;
    int32_t* __restrict__ tile_part;
};
enum { IX_BAD = 1, IX_BITS = 2, IX_POLY = 4, IX_NOT_FIXED = 8, IX_UNALIGNED = 16 };
struct IndexAcc {
    int flags = 0;
    int32_t max_bits = INT32_MIN;
    uint64_t end = 0;
};

// Entry p: its descriptor, the tiles whose last partition it is, and its part
// of the summary.
__device__ __forceinline__ void index_entry(const IndexIn& a, int64_t p, int64_t off, IndexAcc& acc) {
    const int32_t s = a.st[p], e = a.en[p], ty = a.type[p], b = a.bits[p];
    const int32_t len = e > s ? e - s : 0;
    Desc d;
    d.theta0 = a.params[4 * p];
    d.theta1 = a.params[4 * p + 1];
    d.packed = desc_pack(off, b, ty);
    d.start = s;
    d.len = len;
    a.desc[p] = d;
    // validation (sorted, non-overlapping, inside [0, n))
    const bool more = p + 1 < a.P;
    const int32_t s_next = more ? a.st[p + 1] : 0x7FFFFFFF;
    const bool bad = s < 0 || e < s || static_cast<int64_t>(e) > a.n || (more && (e > s_next || s_next < s));
    // fixed-size detection against S = len of partition 0
    const int64_t S = static_cast<int64_t>(a.en[0]) - a.st[0];
    const int64_t fs = S * p;
    const int64_t fe = (fs + S < a.n) ? fs + S : a.n;
    acc.flags |= (bad ? IX_BAD : 0) | ((b < 0 || b > 64) ? IX_BITS : 0) | (ty == MODEL_POLY2 ? IX_POLY : 0) |
                 ((S <= 0 || s != fs || e != fe || (!more && e != a.n)) ? IX_NOT_FIXED : 0) |
                 ((len > 0 && (s % kIndexTile != 0 || (e % kIndexTile != 0 && e != a.n))) ? IX_UNALIGNED : 0);
    acc.max_bits = b > acc.max_bits ? b : acc.max_bits;
    const uint64_t end = static_cast<uint64_t>(off + static_cast<int64_t>(len) * b);  // unsigned, as the atomic
    acc.end = end > acc.end ? end : acc.end;
    // tile_part[t] = last partition with start <= t*1024, for t in [ceil(s/1024), ceil(s_next/1024))
    if (bad) return;
    const int64_t t0 = (p == 0) ? 0 : (static_cast<int64_t>(s) + kIndexTile - 1) >> kIndexShift;
    int64_t t1 = more ? (static_cast<int64_t>(s_next) + kIndexTile - 1) >> kIndexShift : a.n_index;
    if (t1 > a.n_index) t1 = a.n_index;
    for (int64_t t = t0; t < t1; ++t) a.tile_part[t] = static_cast<int32_t>(p);
}

// The workgroup's summary, valid in thread 0 (all threads call it).
__device__ __forceinline__ IndexAcc index_reduce(IndexAcc acc) {
    __shared__ int32_t s_flags[kIndexThreads / 64], s_bits[kIndexThreads / 64];
    __shared__ uint64_t s_end[kIndexThreads / 64];
    int flags = 0;
#pragma unroll
    for (int f = 1; f <= IX_UNALIGNED; f <<= 1) flags |= __any(acc.flags & f) ? f : 0;
    const int32_t wb = wave_max_all(acc.max_bits);
    const uint64_t we = wave_max_all(acc.end);
    if ((threadIdx.x & 63) == 0) {
        s_flags[threadIdx.x >> 6] = flags;
        s_bits[threadIdx.x >> 6] = wb;
        s_end[threadIdx.x >> 6] = we;
    }
    __syncthreads();
    IndexAcc r;
    if (threadIdx.x == 0)
        for (int w = 0; w < kIndexThreads / 64; ++w) {
            r.flags |= s_flags[w];
            r.max_bits = s_bits[w] > r.max_bits ? s_bits[w] : r.max_bits;
            r.end = s_end[w] > r.end ? s_end[w] : r.end;
        }
    return r;
}

// sum is zeroed beforehand.  host: pinned memory that receives the summary
// when the last workgroup is done (no copy to wait for).
__global__ __launch_bounds__(kIndexThreads) void k_build_index(IndexIn a, const int64_t* __restrict__ off,
                                                               IndexSummary* __restrict__ sum,
                                                               IndexSummary* __restrict__ host) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * kIndexThreads + threadIdx.x;
    IndexAcc acc;
    if (p < a.P) index_entry(a, p, off[p], acc);  // every lane stays for the reductions
    const IndexAcc r = index_reduce(acc);
    if (threadIdx.x != 0) return;
    if (r.flags & IX_BAD) atomicOr(&sum->malformed, 1);
    if (r.flags & IX_BITS) atomicOr(&sum->bad_bits, 1);
    if (r.flags & IX_POLY) atomicOr(&sum->has_poly, 1);
    if (r.flags & IX_NOT_FIXED) atomicOr(&sum->not_fixed, 1);
    if (r.flags & IX_UNALIGNED) atomicOr(&sum->unaligned, 1);
    atomicMax(&sum->max_bits, r.max_bits);
    atomicMax(reinterpret_cast<unsigned long long*>(&sum->total_bits), static_cast<unsigned long long>(r.end));
    __threadfence();
    if (atomicAdd(&sum->done, 1) != static_cast<int32_t>(gridDim.x) - 1) return;
    IndexSummary x{};  // the last workgroup: every other one's atomics are done
    x.malformed = atomicOr(&sum->malformed, 0);
    x.bad_bits = atomicOr(&sum->bad_bits, 0);
    x.has_poly = atomicOr(&sum->has_poly, 0);
    x.not_fixed = atomicOr(&sum->not_fixed, 0);
    x.unaligned = atomicOr(&sum->unaligned, 0);
    x.max_bits = atomicMax(&sum->max_bits, INT32_MIN);
    x.total_bits = static_cast<int64_t>(atomicMax(reinterpret_cast<unsigned long long*>(&sum->total_bits), 0ULL));
    *host = x;
}

// The whole index of a small column in one workgroup and one launch: offsets
// (SCAN: from the widths; else given), descriptors, tile_part, summary and tile
// records.  A launch costs 4-5 us with its gap; the six it replaces (three for
// the scan, index, summary clear, tile records) were a quarter of a 2^16-value
// compress.  Limits: beyond kIndexSmall partitions or tiles one workgroup takes
// longer than the launches.
constexpr int64_t kIndexSmall = 4096;
template <bool SCAN>
__global__ __launch_bounds__(kIndexThreads) void k_index_small(IndexIn a, int64_t* __restrict__ off,
                                                               TileInfo* __restrict__ ti,
                                                               IndexSummary* __restrict__ sum,
                                                               IndexSummary* __restrict__ host) {
    __shared__ int64_t s_w[kScanThreads / 64 + 1];
    __shared__ int s_bad;
    static_assert(kIndexThreads == kScanThreads, "one workgroup scans and indexes");
    IndexAcc acc;
    int64_t carry = 0;
    for (int64_t p0 = 0; p0 < a.P; p0 += kIndexThreads) {
        const int64_t p = p0 + threadIdx.x;
        int64_t o = 0;
        if constexpr (SCAN) {
            int64_t tot;
            o = carry + block_excl_scan(p < a.P ? static_cast<int64_t>(a.en[p] - a.st[p]) * a.bits[p] : 0, s_w, &tot);
            carry += tot;
            if (p < a.P) off[p] = o;
        } else if (p < a.P) {
            o = off[p];
        }
        if (p < a.P) index_entry(a, p, o, acc);
    }
    const IndexAcc r = index_reduce(acc);
    if (threadIdx.x == 0) {
        s_bad = r.flags & IX_BAD;
        IndexSummary x{};
        x.malformed = (r.flags & IX_BAD) ? 1 : 0;
        x.bad_bits = (r.flags & IX_BITS) ? 1 : 0;
        x.has_poly = (r.flags & IX_POLY) ? 1 : 0;
        x.not_fixed = (r.flags & IX_NOT_FIXED) ? 1 : 0;
        x.unaligned = (r.flags & IX_UNALIGNED) ? 1 : 0;
        x.max_bits = r.max_bits > 0 ? r.max_bits : 0;
        x.total_bits = static_cast<int64_t>(r.end);
        *sum = x;
        *host = x;
    }
    __threadfence_block();
    __syncthreads();  // descriptors and tile_part of every thread
    if (s_bad) return;  // tile_part is incomplete
    for (int64_t t = threadIdx.x; t < a.n_index - 1; t += kIndexThreads) {
        const int64_t e0 = t * kIndexTile;
        const int64_t e1 = (e0 + kIndexTile < a.n) ? e0 + kIndexTile : a.n;
        ti[t] = make_tile_info(a.desc[a.tile_part[t]], e0, e1);
    }
}

// TileInfo per 1024-element tile (after the descriptors and tile_part exist).
__global__ void k_build_tinfo(const Desc* __restrict__ desc, const int32_t* __restrict__ tile_part, int64_t n,
                              TileInfo* __restrict__ ti, int64_t ntiles) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    const int64_t e0 = t * kIndexTile;
    const int64_t e1 = (e0 + kIndexTile < n) ? e0 + kIndexTile : n;
    ti[t] = make_tile_info(desc[tile_part[t]], e0, e1);
}

// Batched index: descriptors + tile_part for every partition of every column
// (fixed partitions, so always well formed).
__global__ void k_build_index_batch(const BatchCol* __restrict__ cols, const int32_t* __restrict__ part_col,
                                    int64_t Ptot) {
    const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool live = g < Ptot;  // every lane stays for the wave vote below
    const int32_t ci = live ? part_col[g] : -1;
    int32_t b = INT32_MIN;
    if (live) b = cols[ci].bits[g - cols[ci].part_base];
    // a wave whose partitions all belong to one column (the usual case:
    // partitions are consecutive) issues one atomic for that column
    const int32_t c0 = __builtin_amdgcn_readfirstlane(live ? ci : INT32_MAX);
    if (__all(!live || ci == c0)) {
        const int32_t wb = wave_max_all(b);
        if ((threadIdx.x & 63) == 0 && c0 != INT32_MAX) atomicMax(&cols[c0].sum->max_bits, wb);
    } else if (live) {
        atomicMax(&cols[ci].sum->max_bits, b);
    }
    if (!live) return;
    const BatchCol& c = cols[ci];
    const int64_t p = g - c.part_base;
    const int32_t s = c.start[p], e = c.end[p];
    Desc d;
    d.theta0 = c.params[4 * p];
    d.theta1 = c.params[4 * p + 1];
    d.packed = desc_pack(c.off[p], b, c.type[p]);
    d.start = s;
    d.len = e > s ? e - s : 0;
    c.desc[p] = d;
    const int32_t s_next = (p + 1 < c.P) ? c.start[p + 1] : 0x7FFFFFFF;
    const int64_t t0 = (p == 0) ? 0 : (static_cast<int64_t>(s) + kIndexTile - 1) >> kIndexShift;
    int64_t t1 = (p + 1 < c.P) ? (static_cast<int64_t>(s_next) + kIndexTile - 1) >> kIndexShift : c.n_index;
    if (t1 > c.n_index) t1 = c.n_index;
    for (int64_t t = t0; t < t1; ++t) c.tile_part[t] = static_cast<int32_t>(p);
}

// Everything between the fit and the pack of a batch whose columns are small, a
// workgroup per column: offsets, descriptors, tile_part, tile records, summary and
// payload length.  Bound by launches: the five kernels it replaces took 4 to 10 us
// each for little work (1000 columns, 2^26 values in all: 32 -> 14 us, the whole
// compress and decode 341 -> 330; 100 columns, 2^20 values: 69 -> 41 with the fit's
// gains).  Beyond kBatchSmall partitions or tiles in one column its workgroup would
// take longer than the launches.
constexpr int kBatchIndexThreads = 256;
constexpr int64_t kBatchSmall = 2048;
__global__ __launch_bounds__(kBatchIndexThreads) void k_batch_index(BatchCol* __restrict__ cols,
                                                                    int64_t* __restrict__ col_bits) {
    __shared__ int64_t s_w[kBatchIndexThreads / 64 + 1];
    __shared__ int32_t s_max[kBatchIndexThreads / 64];
    const BatchCol c = cols[blockIdx.x];
    const int tid = threadIdx.x;
    int64_t carry = 0;
    int32_t max_bits = 0;
    for (int64_t p0 = 0; p0 < c.P; p0 += kBatchIndexThreads) {
        const int64_t p = p0 + tid;
        const bool in = p < c.P;
        const int32_t st = in ? c.start[p] : 0, en = in ? c.end[p] : 0, b = in ? c.bits[p] : 0;
        int64_t tot;
        const int64_t off =
            carry + block_excl_scan<kBatchIndexThreads>(static_cast<int64_t>(en - st) * b, s_w, &tot);
        carry += tot;
        max_bits = b > max_bits ? b : max_bits;
        if (!in) continue;
        c.off[p] = off;
        Desc d;
        d.theta0 = c.params[4 * p];
        d.theta1 = c.params[4 * p + 1];
        d.packed = desc_pack(off, b, c.type[p]);
        d.start = st;
        d.len = en > st ? en - st : 0;
        c.desc[p] = d;
        // as in k_build_index_batch; partition p + 1 starts where p ends
        const int64_t t0 = p == 0 ? 0 : (static_cast<int64_t>(st) + kIndexTile - 1) >> kIndexShift;
        int64_t t1 = p + 1 < c.P ? (static_cast<int64_t>(en) + kIndexTile - 1) >> kIndexShift : c.n_index;
        if (t1 > c.n_index) t1 = c.n_index;
        for (int64_t t = t0; t < t1; ++t) c.tile_part[t] = static_cast<int32_t>(p);
    }
    max_bits = wave_max_all(max_bits);
    if ((tid & 63) == 0) s_max[tid >> 6] = max_bits;
    __threadfence_block();
    __syncthreads();  // descriptors and tile_part of every thread
    if (tid == 0) {
        IndexSummary x{};
        for (int k = 0; k < kBatchIndexThreads / 64; ++k) x.max_bits = s_max[k] > x.max_bits ? s_max[k] : x.max_bits;
        const int64_t w = (carry + 31) / 32;
        x.bad_bits = w > c.words_reserved ? 1 : 0;  // cannot happen: reserve is the worst case
        *c.sum = x;
        cols[blockIdx.x].payload_words = w;
        col_bits[blockIdx.x] = carry;
    }
    for (int64_t t = tid; t * kIndexTile < c.n; t += kBatchIndexThreads) {
        const int64_t e0 = t * kIndexTile;
        const int64_t e1 = (e0 + kIndexTile < c.n) ? e0 + kIndexTile : c.n;
        c.tinfo[t] = make_tile_info(c.desc[c.tile_part[t]], e0, e1);
    }
}

__global__ void k_build_tinfo_batch(const BatchCol* __restrict__ cols, const int32_t* __restrict__ tile_col,
                                    int64_t Ttot) {
    const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= Ttot) return;
    const BatchCol& c = cols[tile_col[g]];
    const int64_t t = g - c.tile_base;
    const int64_t e0 = t * kIndexTile;
    const int64_t e1 = (e0 + kIndexTile < c.n) ? e0 + kIndexTile : c.n;
    c.tinfo[t] = make_tile_info(c.desc[c.tile_part[t]], e0, e1);
}

// ---------------------------------------------------------------------------
// Pack, one wave per 1024-value tile.  Tiles inside one partition: word-major
// (pack_wave).  Other tiles: the codes are ORed into the tile's words in LDS
// (pack_span).
// ---------------------------------------------------------------------------
// bit position of element e's first bit, or of the next stored bit when e is
// in a gap / past the end of the last partition with start <= e.
__device__ __forceinline__ int64_t bitpos_lb(const Desc* __restrict__ desc, int64_t plo, int64_t phi, int64_t e) {
    // last partition in [plo, phi] with start <= e
    int64_t lo = plo, hi = phi;
    while (lo < hi) {
        int64_t m = (lo + hi + 1) >> 1;
        if (desc[m].start <= e) lo = m; else hi = m - 1;
    }
    const Desc d = desc[lo];
    if (e < d.start) return desc_off(d.packed);
    int64_t k = e - d.start;
    if (k > d.len) k = d.len;
    return desc_off(d.packed) + k * desc_bits(d.packed);
}

// Wave pack of one 1024-value tile that lies inside one partition (the
// tile's TileInfo path is not TILE_SLOW).  Phase 1: coalesced loads, one
// residual code per value (lane l: values l, l+64, ...), parked in the
// wave's LDS slice.  Phase 2, word-major: lane j assembles output words j,
// j+64, ... from the (at most 32/bits + 2) codes that overlap each word, so
// no word is shared between lanes and no atomics are needed inside the
// tile.  Every word the tile covers completely is stored whole.  A word the
// tile starts or ends inside is shared with the neighbouring tile; its
// partial value is returned as an edge (wave-uniform) for merge_edges.
// EDGES = false: a column without partition-spanning tiles.  Its partitions
// start on tiles and its tiles hold 1024 * bits bits, so every tile starts on a
// word and only the column's last word can be partial, with nothing after it:
// every word is stored whole, nothing has to be zeroed or merged.
constexpr int kPackWaves = 4;

struct PackEdge {
    uint32_t* p;  // nullptr: no partial word
    uint32_t v;
};

template <class T, bool EDGES>
__device__ __forceinline__ void pack_wave(const T* __restrict__ v, const Desc* __restrict__ desc, const TileInfo& x,
                                          int64_t e0, int64_t e1, uint32_t* __restrict__ words, int lane,
                                          uint64_t* __restrict__ s_code, PackEdge& ef, PackEdge& el) {
    ef = PackEdge{nullptr, 0};
    el = PackEdge{nullptr, 0};
    const int b = tile_bits(x.info);
    if (b == 0) return;
    const bool direct = tile_type(x.info) == MODEL_DIRECT_COPY;
    const int32_t lbase = x.lbase;
    const int32_t cnt = static_cast<int32_t>(e1 - e0);
    const uint64_t mask = (b < 64) ? ((1ULL << b) - 1ULL) : ~0ULL;
    const T* __restrict__ vt = v + e0;
    T val[kIndexTile / 64];
#pragma unroll
    for (int r = 0; r < kIndexTile / 64; ++r) {  // all 16 loads in flight before any compute
        const int32_t k = r * 64 + lane;
        val[r] = vt[k < cnt ? k : cnt - 1];
    }
    // Tiles whose predictions need no saturation (the common case) take the
    // branch-free residual; the codes are the same either way.
    const int tier = direct ? 0
                            : enc_tier<T>(__builtin_fma(x.t1, static_cast<double>(lbase), x.t0),
                                          __builtin_fma(x.t1, static_cast<double>(lbase + cnt - 1), x.t0));
    if (tier == 1) {
#pragma unroll
        for (int r = 0; r < kIndexTile / 64; ++r) {
            const int32_t k = r * 64 + lane;
            const uint64_t code = static_cast<uint64_t>(enc_delta_fast<T, 1>(val[r], x.t0, x.t1, lbase + k));
            s_code[k] = (k < cnt) ? (code & mask) : 0;
        }
    } else if (std::is_same<T, int64_t>::value && tier == 2) {
#pragma unroll
        for (int r = 0; r < kIndexTile / 64; ++r) {
            const int32_t k = r * 64 + lane;
            const uint64_t code = static_cast<uint64_t>(enc_delta_fast<T, 2>(val[r], x.t0, x.t1, lbase + k));
            s_code[k] = (k < cnt) ? (code & mask) : 0;
        }
    } else {
#pragma unroll
        for (int r = 0; r < kIndexTile / 64; ++r) {
            const int32_t k = r * 64 + lane;
            const uint64_t code =
                direct ? static_cast<uint64_t>(val[r])
                       : static_cast<uint64_t>(calc_delta<T>(val[r], enc_pred<T>(x.t0, x.t1, lbase + k)));
            s_code[k] = (k < cnt) ? (code & mask) : 0;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int64_t w0 = x.W >> 5;
    const int32_t r0 = static_cast<int32_t>(x.W & 31);
    const int32_t Wt = (r0 + cnt * b + 31) >> 5;  // <= 2049
    // floor(y / b) as mul_hi(y, ceil(2^32 / b)): exact for y * b < 2^32, and
    // here y <= 32 * 2049 + 31 < 2^17 with b <= 64.
    const uint32_t rcp = 0xFFFFFFFFu / static_cast<uint32_t>(b) + 1u;
    const auto div_b = [&](int32_t y) -> int32_t {
        return b == 1 ? y : static_cast<int32_t>(__umulhi(static_cast<uint32_t>(y), rcp));
    };
    const bool start_partial = r0 != 0;
    const bool end_partial = ((r0 + cnt * b) & 31) != 0;
    uint32_t vf = 0, vl = 0;
    for (int32_t j = lane; j < Wt; j += 64) {
        const int32_t lo_bit = 32 * j - r0;  // first stream bit of word j (relative to element e0)
        const int32_t k0 = lo_bit < 0 ? 0 : div_b(lo_bit);
        int32_t k1 = div_b(lo_bit + 31);
        if (k1 > cnt - 1) k1 = cnt - 1;
        uint32_t wv = 0;
        for (int32_t k = k0; k <= k1; ++k) {
            const uint64_t code = s_code[k];
            const int32_t pos = k * b - lo_bit;  // in (-b, 32)
            wv |= (pos >= 0) ? static_cast<uint32_t>(code << pos) : static_cast<uint32_t>(code >> (-pos));
        }
        if (EDGES && j == 0 && start_partial) vf = wv;
        else if (EDGES && j == Wt - 1 && end_partial) vl = wv;
        else words[w0 + j] = wv;
    }
    if constexpr (!EDGES) return;
    // word 0 is lane 0's first word; word Wt - 1 is lane (Wt - 1) % 64's last
    if (start_partial) ef = PackEdge{words + w0, static_cast<uint32_t>(__builtin_amdgcn_readlane(vf, 0))};
    if (end_partial && !(start_partial && Wt == 1))
        el = PackEdge{words + w0 + Wt - 1, static_cast<uint32_t>(__builtin_amdgcn_readlane(vl, (Wt - 1) & 63))};
}

// The partial words of a workgroup's tiles, in bit order (first and last
// edge of each wave).  Two entries with the same word can only be adjacent
// (non-empty tiles of 1024 values span at least 32 bits); such a pair is the
// word's whole content and is stored plainly.  The first and last entries
// may share their word with a tile of another workgroup: OR-ed atomically.
// Any other unpaired entry shares its word only with a tile of the
// partition-spanning path, whose own kernel runs later and ORs its part in
// atomically, so a plain store is correct there too.  One thread.
__device__ __forceinline__ void merge_edges(const PackEdge* __restrict__ e, int m) {
    int first = -1, last = -1;
    for (int k = 0; k < m; ++k)
        if (e[k].p) {
            if (first < 0) first = k;
            last = k;
        }
    if (first < 0) return;
    int k = first;
    while (k <= last) {
        uint32_t* p = e[k].p;
        uint32_t v = e[k].v;
        bool outer = k == first;
        int k2 = k + 1;
        while (k2 <= last && !e[k2].p) ++k2;
        if (k2 <= last && e[k2].p == p) {
            v |= e[k2].v;
            outer = outer || k2 == last;
            k2 += 1;
            while (k2 <= last && !e[k2].p) ++k2;
        } else {
            outer = outer || k == last;
        }
        if (outer) {
            if (v) atomicOr(p, v);
        } else {
            *p = v;
        }
        k = k2;
    }
}

template <class T, bool EDGES>
__global__ __launch_bounds__(64 * kPackWaves) void k_pack_wave(const T* __restrict__ v, const Desc* __restrict__ desc,
                                                               const TileInfo* __restrict__ tinfo, int64_t n,
                                                               uint32_t* __restrict__ words) {
    __shared__ uint64_t s_code[kPackWaves][kIndexTile];
    __shared__ PackEdge s_edge[2 * kPackWaves];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kPackWaves + wave;
    const int64_t e0 = t * kIndexTile;
    PackEdge ef{nullptr, 0}, el{nullptr, 0};
    if (e0 < n) {
        const TileInfo x = tinfo[t];
        if (tile_path(x.info) != TILE_SLOW) {
            const int64_t e1 = (e0 + kIndexTile < n) ? e0 + kIndexTile : n;
            pack_wave<T, EDGES>(v, desc, x, e0, e1, words, lane, s_code[wave], ef, el);
        }
    }
    if constexpr (!EDGES) return;
    if (lane == 0) {
        s_edge[2 * wave] = ef;
        s_edge[2 * wave + 1] = el;
    }
    __syncthreads();
    if (threadIdx.x == 0) merge_edges(s_edge, 2 * kPackWaves);
}

// Pack of one tile of the partition-spanning path by a wave: a value per lane
// and row, its partition from the staged map (a search over the tile's candidates
// where that does not apply), its code ORed into the tile's words in LDS (a
// tile's bits are contiguous: gaps and empty partitions store none), then the
// words stored in order.  A first or last word that the tile does not fill is
// returned as an edge (wave-uniform); a tile inside one word that continues on
// both sides returns that word twice, the second time empty.  2e7 int64 values in
// partitions of 1000: 63.5 us where a workgroup per tile with a search per
// value took 130 us; instructions bound it (uint32, half the bytes: 51 us).
// Values are loaded at once and packed kSpanRows rows at a time, the last
// partial word carried over, so that a wave needs 5 KB of LDS (the whole tile's
// words would take 11 and leave 3 waves per SIMD: 97 us).
constexpr int kSpanRows = 4;
constexpr int kSpanWords = 2 * 64 * kSpanRows + 4;  // 64-bit fields from any bit of the first word on

// A partition as pack_span takes it, relative to the tile: value x of the tile
// is the partition's value x - sx and its first bit is bit off + x * bits from the
// tile's first word on (mod 2^32; a tile has at most 2^16 bits).  32-bit index and
// bit arithmetic and the branch-free residual where the whole partition allows
// it: 63.5 us where the same loop on Desc took 75.
struct alignas(16) SpanDesc {
    double t0, t1;
    int32_t sx;
    uint32_t len;
    uint32_t off;
    int32_t info;  // bits | DIRECT_COPY << 8 | tier 1 of enc_tier << 9
};
struct SpanMap {
    SpanDesc d[kManyParts];
    uint32_t bits[kManyBits];
};

template <class T> __device__ __forceinline__ SpanDesc span_desc(const Desc& d, int64_t e0, int64_t W0) {
    const int b = desc_bits(d.packed);
    const int32_t sx = static_cast<int32_t>(d.start - e0);  // > -2^31: starts are int32 >= 0
    const bool direct = desc_type(d.packed) == MODEL_DIRECT_COPY;
    const bool fast = !direct && d.len > 0 && fit_tier<T>(d.len, d.theta0, d.theta1) == 1;
    return SpanDesc{d.theta0, d.theta1, sx, static_cast<uint32_t>(d.len),
                    static_cast<uint32_t>(desc_off(d.packed) - (W0 & ~31LL)) -
                        static_cast<uint32_t>(sx) * static_cast<uint32_t>(b),
                    b | (direct ? 256 : 0) | (fast ? 512 : 0)};
}

template <class T>
__device__ __forceinline__ void pack_span(const T* __restrict__ v, const Desc* __restrict__ desc,
                                          const int32_t* __restrict__ tile_part, int64_t e0, int64_t e1,
                                          uint32_t* __restrict__ words, int lane, SpanMap& L, uint32_t* s_w,
                                          PackEdge& ef, PackEdge& el) {
    ef = PackEdge{nullptr, 0};
    el = PackEdge{nullptr, 0};
    const int32_t cnt = static_cast<int32_t>(e1 - e0);
    const T* __restrict__ vt = v + e0;
    T val[kIndexTile / 64];
#pragma unroll
    for (int r = 0; r < kIndexTile / 64; ++r) {
        const int32_t x = r * 64 + lane;
        val[r] = vt[x < cnt ? x : cnt - 1];
    }
    const int64_t plo = tile_part[e0 >> kIndexShift];
    const int64_t phi = tile_part[(e1 + kIndexTile - 1) >> kIndexShift];
    const int64_t W0 = bitpos_lb(desc, plo, plo, e0);
    const bool mapped = phi - plo < kManyParts &&
                        many_stage(plo, static_cast<int>(phi - plo + 1), lane, L.bits, [&](int64_t p, int i) {
                            const SpanDesc d = span_desc<T>(desc[p], e0, W0);
                            L.d[i] = d;
                            return d.sx;
                        });
    int base = 0;
    uint32_t* __restrict__ out = words + (W0 >> 5);  // word of s_w[0]
    uint32_t done = 0;                               // bits of the tile's words stored so far
    int32_t used = static_cast<int32_t>(W0 & 31);    // bits of s_w[0] before this step's
    uint32_t carry = 0;                              // and their value, of this tile's own bits
    bool first = used != 0;                          // s_w[0] is the tile's partial first word
#pragma unroll
    for (int r0 = 0; r0 < kIndexTile / 64; r0 += kSpanRows) {
        for (int i = lane; i < kSpanWords; i += 64) s_w[i] = i == 0 ? carry : 0;
        wave_lds_fence();
        int32_t end = used;  // bits used, from s_w[0]'s bit 0
#pragma unroll
        for (int k = 0; k < kSpanRows; ++k) {
            const int32_t x = (r0 + k) * 64 + lane;
            SpanDesc d;
            if (mapped) {
                d = L.d[many_index(L.bits, r0 + k, lane, base)];
            } else {
                int64_t lo = plo, hi = phi;
                while (lo < hi) {
                    const int64_t m = (lo + hi + 1) >> 1;
                    if (desc[m].start <= e0 + x) lo = m; else hi = m - 1;
                }
                d = span_desc<T>(desc[lo], e0, W0);
            }
            const int b = d.info & 255;
            const int32_t i = x - d.sx;
            if (x >= cnt || static_cast<uint32_t>(i) >= d.len || b == 0) continue;
            uint64_t code;
            if (d.info & 512) code = static_cast<uint64_t>(enc_delta_fast<T>(val[r0 + k], d.t0, d.t1, i));
            else if (d.info & 256) code = static_cast<uint64_t>(val[r0 + k]);
            else code = static_cast<uint64_t>(calc_delta<T>(val[r0 + k], enc_pred<T>(d.t0, d.t1, i)));
            const uint32_t rel = d.off + static_cast<uint32_t>(x) * static_cast<uint32_t>(b) - done;
            const uint32_t wi = rel >> 5, sh = rel & 31;
            if (b <= 32) {
                const uint32_t c = static_cast<uint32_t>(code) & (0xFFFFFFFFu >> (32 - b));
                atomicOr(&s_w[wi], c << sh);
                if (sh + b > 32) atomicOr(&s_w[wi + 1], c >> (32 - sh));
            } else {
                if (b < 64) code &= (1ULL << b) - 1ULL;
                atomicOr(&s_w[wi], static_cast<uint32_t>(code << sh));
                if (sh + b > 32) atomicOr(&s_w[wi + 1], static_cast<uint32_t>(code >> (32 - sh)));
                if (sh + b > 64) atomicOr(&s_w[wi + 2], static_cast<uint32_t>(code >> (64 - sh)));
            }
            end = static_cast<int32_t>(rel) + b;  // increases along a lane's values
        }
        for (int o = 32; o > 0; o >>= 1) {
            const int32_t y = __shfl_xor(end, o, 64);
            end = y > end ? y : end;
        }
        wave_lds_fence();
        const int32_t full = end >> 5;  // words complete after this step
        for (int32_t j = lane; j < full; j += 64)
            if (j > 0 || !first) out[j] = s_w[j];
        if (full > 0 && first) {
            ef = PackEdge{out, s_w[0]};
            first = false;
        }
        carry = s_w[full];
        used = end & 31;
        out += full;
        done += static_cast<uint32_t>(full) << 5;
        wave_lds_fence();  // s_w is the next rows'
    }
    // the word the tile ends inside (a tile may also begin inside it)
    if (used == 0) return;
    if (first) {
        if (used == (W0 & 31)) return;  // nothing stored
        ef = PackEdge{out, carry};
        carry = 0;
    }
    el = PackEdge{out, carry};
}

// The edges of a workgroup's spanning tiles (first and last of each tile, in
// bit order; null where there is none).  A run of equal words is the word's
// whole content when it begins with a tile's last word and ends with a tile's
// first one, and is stored; every other word has more bits in another tile (of
// another workgroup, or packed by k_pack_wave before) and is ORed.  One thread.
__device__ __forceinline__ void merge_span_edges(const PackEdge* __restrict__ e, int m) {
    int k = 0;
    while (k < m) {
        if (!e[k].p) {
            ++k;
            continue;
        }
        uint32_t v = e[k].v;
        const bool from_last = (k & 1) != 0;
        int last = k, q = k + 1;
        for (; q < m; ++q) {
            if (!e[q].p) continue;
            if (e[q].p != e[k].p) break;
            v |= e[q].v;
            last = q;
        }
        if (from_last && !(last & 1)) *e[k].p = v;
        else if (v) atomicOr(e[k].p, v);
        k = q;
    }
}

struct SpanLds {
    SpanMap many[kPackWaves];
    uint32_t w[kPackWaves][kSpanWords];
    PackEdge edge[2 * kPackWaves];
};

template <class T>
__global__ __launch_bounds__(64 * kPackWaves) void k_pack_span(const T* __restrict__ v, const Desc* __restrict__ desc,
                                                               const int32_t* __restrict__ tile_part,
                                                               const TileInfo* __restrict__ tinfo, int64_t n,
                                                               uint32_t* __restrict__ words) {
    __shared__ SpanLds S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kPackWaves + wave;
    const int64_t e0 = t * kIndexTile;
    PackEdge ef{nullptr, 0}, el{nullptr, 0};
    if (e0 < n && tile_path(tinfo[t].info) == TILE_SLOW) {
        const int64_t e1 = (e0 + kIndexTile < n) ? e0 + kIndexTile : n;
        pack_span<T>(v, desc, tile_part, e0, e1, words, lane, S.many[wave], S.w[wave], ef, el);
    }
    if (lane == 0) {
        S.edge[2 * wave] = ef;
        S.edge[2 * wave + 1] = el;
    }
    __syncthreads();
    if (threadIdx.x == 0) merge_span_edges(S.edge, 2 * kPackWaves);
}

// Batched wave pack over the 1024-value tiles of every column, every element
// type in one launch (the type comes from the column); tiles that span
// partitions are left to k_pack_span_batch.
template <bool EDGES>
__global__ __launch_bounds__(64 * kPackWaves) void k_pack_wave_batch(const BatchCol* __restrict__ cols,
                                                                     const int32_t* __restrict__ tile_col, int64_t Ttot) {
    __shared__ uint64_t s_code[kPackWaves][kIndexTile];
    __shared__ PackEdge s_edge[2 * kPackWaves];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t g = static_cast<int64_t>(blockIdx.x) * kPackWaves + wave;
    PackEdge ef{nullptr, 0}, el{nullptr, 0};
    if (g < Ttot) {
        const BatchCol& c = cols[tile_col[g]];
        if (c.payload_words <= c.words_reserved) {
            const int64_t t = g - c.tile_base;
            const TileInfo x = c.tinfo[t];
            if (tile_path(x.info) != TILE_SLOW) {
                const int64_t e0 = t * kIndexTile;
                const int64_t e1 = (e0 + kIndexTile < c.n) ? e0 + kIndexTile : c.n;
                switch (c.dtype) {
                    case GLC_I32:
                        pack_wave<int32_t, EDGES>(static_cast<const int32_t*>(c.values), c.desc, x, e0, e1, c.words, lane,
                                           s_code[wave], ef, el);
                        break;
                    case GLC_U32:
                        pack_wave<uint32_t, EDGES>(static_cast<const uint32_t*>(c.values), c.desc, x, e0, e1, c.words, lane,
                                            s_code[wave], ef, el);
                        break;
                    case GLC_I64:
                        pack_wave<int64_t, EDGES>(static_cast<const int64_t*>(c.values), c.desc, x, e0, e1, c.words, lane,
                                           s_code[wave], ef, el);
                        break;
                    default:
                        pack_wave<uint64_t, EDGES>(static_cast<const uint64_t*>(c.values), c.desc, x, e0, e1, c.words, lane,
                                            s_code[wave], ef, el);
                        break;
                }
            }
        }
    }
    if constexpr (!EDGES) return;
    // tiles of different columns never share a word (separate payloads), so
    // their edges never pair
    if (lane == 0) {
        s_edge[2 * wave] = ef;
        s_edge[2 * wave + 1] = el;
    }
    __syncthreads();
    if (threadIdx.x == 0) merge_edges(s_edge, 2 * kPackWaves);
}

// The spanning tiles of every column of a batch.
__global__ __launch_bounds__(64 * kPackWaves) void k_pack_span_batch(const BatchCol* __restrict__ cols,
                                                                     const int32_t* __restrict__ tile_col, int64_t Ttot) {
    __shared__ SpanLds S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t g = static_cast<int64_t>(blockIdx.x) * kPackWaves + wave;
    PackEdge ef{nullptr, 0}, el{nullptr, 0};
    if (g < Ttot) {
        const BatchCol& c = cols[tile_col[g]];
        const int64_t t = g - c.tile_base;
        if (c.payload_words <= c.words_reserved && tile_path(c.tinfo[t].info) == TILE_SLOW) {
            const int64_t e0 = t * kIndexTile;
            const int64_t e1 = (e0 + kIndexTile < c.n) ? e0 + kIndexTile : c.n;
            switch (c.dtype) {
                case GLC_I32:
                    pack_span<int32_t>(static_cast<const int32_t*>(c.values), c.desc, c.tile_part, e0, e1, c.words, lane,
                                       S.many[wave], S.w[wave], ef, el);
                    break;
                case GLC_U32:
                    pack_span<uint32_t>(static_cast<const uint32_t*>(c.values), c.desc, c.tile_part, e0, e1, c.words,
                                        lane, S.many[wave], S.w[wave], ef, el);
                    break;
                case GLC_I64:
                    pack_span<int64_t>(static_cast<const int64_t*>(c.values), c.desc, c.tile_part, e0, e1, c.words, lane,
                                       S.many[wave], S.w[wave], ef, el);
                    break;
                default:
                    pack_span<uint64_t>(static_cast<const uint64_t*>(c.values), c.desc, c.tile_part, e0, e1, c.words,
                                        lane, S.many[wave], S.w[wave], ef, el);
                    break;
            }
        }
    }
    // tiles of different columns never share a word (separate payloads)
    if (lane == 0) {
        S.edge[2 * wave] = ef;
        S.edge[2 * wave + 1] = el;
    }
    __syncthreads();
    if (threadIdx.x == 0) merge_span_edges(S.edge, 2 * kPackWaves);
}

// ---------------------------------------------------------------------------
// V6 partitioner
// ---------------------------------------------------------------------------
constexpr int kV6Threads = 128;  // compression/GpuPartitioner.cuh:53

template <class T>
__global__ __launch_bounds__(kV6Threads) void k_v6_var(const T* __restrict__ v, int64_t n, int64_t vbs,
                                                       int64_t nvb, float* __restrict__ var) {
    __shared__ float s_stat[4];
    const int tid = threadIdx.x;
    for (int64_t blk = blockIdx.x; blk < nvb; blk += gridDim.x) {
        const int64_t s = blk * vbs;
        const int64_t e = (s + vbs < n) ? s + vbs : n;
        const double dn = static_cast<double>(e - s);
        double sum = 0.0, ssq = 0.0, c1 = 0.0, c2 = 0.0;
        // Kahan, PartitioningKernels.cuh:669-682, over i = s + tid, s + tid +
        // 128, ... in that order; eight loads per thread in flight together
        // (branch-free, the index clamped to e - 1).
        for (int64_t base = s; base < e; base += 8 * kV6Threads) {
            T y[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int64_t i = base + k * kV6Threads + tid;
                y[k] = v[i < e ? i : e - 1];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (base + k * kV6Threads + tid < e) {
                    const double val = static_cast<double>(y[k]);
                    const double y1 = val - c1;
                    const double t1 = sum + y1;
                    c1 = (t1 - sum) - y1;
                    sum = t1;
                    const double y2 = __builtin_fma(val, val, -c2);
                    const double t2 = ssq + y2;
                    c2 = (t2 - ssq) - y2;
                    ssq = t2;
                }
            }
        }
        for (int o = 16; o > 0; o >>= 1) {  // 32-lane tree of MathHelpers.cuh:91-95
            sum = sum + __shfl_down(sum, o, 32);
            ssq = ssq + __shfl_down(ssq, o, 32);
        }
        if ((tid & 31) == 0) {
            const double q = sum / dn;
            s_stat[tid >> 5] = static_cast<float>(__builtin_fma(-q, q, ssq / dn));
        }
        __syncthreads();
        if (tid == 0) {
            float acc = 0.0f;
            for (int w = 0; w < 4; ++w) acc = acc + s_stat[w];
            var[blk] = acc;
        }
        __syncthreads();
    }
}

__device__ __forceinline__ uint32_t float_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_float(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k;
    return __uint_as_float(u);
}

// Order statistics sorted[nvb/4], sorted[nvb/2], sorted[3nvb/4] by 4-pass
// radix selection on 8-bit digits of the order-preserving key (one
// workgroup; the reference sorts with thrust::sort).  The three ranks are
// selected together: pass 0 builds one histogram (every prefix is empty),
// later passes one per rank.  Wave q finds rank q's digit with a 64-lane
// scan of the 256 bins (4 per lane).  Keys stay in registers when
// nvb <= 1024 * kSelKeys.
constexpr int kSelKeys = 16;

// Lanes of a wave that count in the same bin add once: the leading digits of
// the statistics are nearly all alike, and 16384 LDS atomics on a few addresses
// were most of the selection's 34 us.  Two rounds take the common digits; what is
// left counts lane by lane.
__device__ __forceinline__ void hist_add(uint32_t* hist, uint32_t d, bool on) {
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        const uint64_t m = __ballot(on);
        if (m == 0) return;
        const uint32_t lead = __shfl(d, __builtin_ctzll(m), 64);
        const uint64_t same = __ballot(on && d == lead);
        if ((threadIdx.x & 63) == __builtin_ctzll(m)) atomicAdd(&hist[lead], static_cast<uint32_t>(__popcll(same)));
        on = on && d != lead;
    }
    if (on) atomicAdd(&hist[d], 1u);
}

// All lanes call it; live: the lane holds a key.
__device__ __forceinline__ void sel_count(uint32_t k, bool live, int pass, uint32_t hmask, int shift,
                                          const uint32_t* pre, uint32_t (*hist)[256]) {
    const uint32_t d = (k >> shift) & 0xFFu;
    if (pass == 0) {
        hist_add(hist[0], d, live);
        return;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) hist_add(hist[q], d, live && (k & hmask) == pre[q]);
}

// thr (LDS) is complete after the caller's next barrier.
__device__ __forceinline__ void v6_select(const float* __restrict__ var, int64_t nvb, float (&thr)[3]) {
    __shared__ uint32_t hist[3][256];
    __shared__ uint32_t s_prefix[3];
    __shared__ int64_t s_rank[3];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const bool in_regs = nvb <= 1024LL * kSelKeys;
    uint32_t keys[kSelKeys];
    if (in_regs) {
#pragma unroll
        for (int k = 0; k < kSelKeys; ++k) {
            const int64_t i = tid + 1024LL * k;
            keys[k] = float_key(var[i < nvb ? i : nvb - 1]);
        }
    }
    if (tid < 3) {
        s_prefix[tid] = 0;
        s_rank[tid] = (tid == 0) ? nvb / 4 : (tid == 1) ? nvb / 2 : 3 * nvb / 4;
    }
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        const uint32_t hmask = (pass == 0) ? 0u : (0xFFFFFFFFu << (32 - 8 * pass));
        if (tid < 3 * 256) (&hist[0][0])[tid] = 0;
        __syncthreads();
        const uint32_t pre[3] = {s_prefix[0], s_prefix[1], s_prefix[2]};
        if (in_regs) {
#pragma unroll
            for (int k = 0; k < kSelKeys; ++k) {
                if (1024LL * k >= nvb) break;  // uniform
                sel_count(keys[k], tid + 1024LL * k < nvb, pass, hmask, shift, pre, hist);
            }
        } else {
            for (int64_t i0 = 0; i0 < nvb; i0 += 1024) {
                const int64_t i = i0 + tid;
                sel_count(float_key(var[i < nvb ? i : nvb - 1]), i < nvb, pass, hmask, shift, pre, hist);
            }
        }
        __syncthreads();
        if (wave < 3) {
            const uint32_t* h = hist[pass == 0 ? 0 : wave];
            const uint32_t h0 = h[4 * lane], h1 = h[4 * lane + 1], h2 = h[4 * lane + 2], h3 = h[4 * lane + 3];
            const uint32_t sum = h0 + h1 + h2 + h3;
            uint32_t incl = sum;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(incl, o, 64);
                if (lane >= o) incl += y;
            }
            const int64_t excl = static_cast<int64_t>(incl) - sum;
            const int64_t r = s_rank[wave];
            // the first digit whose running count exceeds r
            if (r >= excl && r < static_cast<int64_t>(incl)) {
                int64_t rr = r - excl;
                uint32_t d = 4 * lane;
                if (rr >= h0) {
                    rr -= h0; ++d;
                    if (rr >= h1) {
                        rr -= h1; ++d;
                        if (rr >= h2) { rr -= h2; ++d; }
                    }
                }
                s_rank[wave] = rr;
                s_prefix[wave] = pre[wave] | (d << shift);
            }
        }
        __syncthreads();
    }
    if (tid < 3) thr[tid] = key_float(s_prefix[tid]);
}
__global__ __launch_bounds__(1024) void k_v6_select(const float* __restrict__ var, int64_t nvb,
                                                    float* __restrict__ thr) {
    __shared__ float s_thr[3];
    v6_select(var, nvb, s_thr);
    if (threadIdx.x < 3) thr[threadIdx.x] = s_thr[threadIdx.x];  // each its own
}

struct V6Count {
    const float* var;
    const float* thr;
    int64_t vbs, n;
    int32_t base;
    __device__ int64_t size_of(int64_t b) const {  // PartitioningKernels.cuh:722-731
        const float x = var[b];
        return x < thr[0] ? 4LL * base : x < thr[1] ? 2LL * base : x < thr[2] ? base : base / 2;
    }
    __device__ int64_t operator()(int64_t b) const {
        const int64_t s = b * vbs;
        const int64_t e = (s + vbs < n) ? s + vbs : n;
        const int64_t sz = size_of(b);
        return (e - s + sz - 1) / sz;
    }
};

// Block b's partitions from entry k on.
__device__ __forceinline__ void v6_emit(const V6Count& f, int64_t b, int64_t k, int32_t* __restrict__ st,
                                        int32_t* __restrict__ en) {
    const int64_t s = b * f.vbs;
    const int64_t e = (s + f.vbs < f.n) ? s + f.vbs : f.n;
    const int64_t sz = f.size_of(b);
    for (int64_t j = s; j < e; j += sz, ++k) {  // PartitioningKernels.cuh:734-741
        st[k] = static_cast<int32_t>(j);
        en[k] = static_cast<int32_t>((j + sz < f.n) ? j + sz : f.n);
    }
}

// host (pinned, or null): the number of partitions and the first one's length
__device__ __forceinline__ void v6_report(const V6Count& f, int64_t total, int64_t* __restrict__ host) {
    const int64_t sz = f.size_of(0);
    host[0] = total;
    host[1] = sz < f.n ? sz : f.n;
}

__global__ void k_v6_emit(V6Count f, int64_t nvb, const int64_t* __restrict__ base_idx, int32_t* __restrict__ st,
                          int32_t* __restrict__ en, const int64_t* __restrict__ total, int64_t* __restrict__ host) {
    const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b == 0 && host) v6_report(f, *total, host);
    if (b < nvb) v6_emit(f, b, base_idx[b], st, en);
}

// Thresholds, counts and partitions of a short list of blocks in one
// workgroup: one launch instead of five.  Up to kV6Small blocks (2^25 values at
// the default base); beyond, writing 16 partitions a block from one workgroup
// takes longer than the launches.
constexpr int64_t kV6Small = 2048;
__global__ __launch_bounds__(1024) void k_v6_small(V6Count f, int64_t nvb, int32_t* __restrict__ st,
                                                   int32_t* __restrict__ en, int64_t* __restrict__ total,
                                                   int64_t* __restrict__ host) {
    __shared__ int64_t s_w[kScanThreads / 64 + 1];
    __shared__ float s_thr[3];
    v6_select(f.var, nvb, s_thr);
    __syncthreads();
    f.thr = s_thr;
    int64_t carry = 0;
    for (int64_t b0 = 0; b0 < nvb; b0 += 1024) {
        const int64_t b = b0 + threadIdx.x;
        int64_t tot;
        const int64_t k = carry + block_excl_scan(b < nvb ? f(b) : 0, s_w, &tot);
        carry += tot;
        if (b < nvb) v6_emit(f, b, k, st, en);
    }
    if (threadIdx.x == 0) {
        *total = carry;
        if (host) v6_report(f, carry, host);
    }
}

__global__ void k_fill_u32(uint32_t* p, int64_t n, uint32_t v) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[i] = v;
}

template <class F> int dispatch_dtype(int dtype, F&& f) {
    switch (dtype) {
        case GLC_I32: return f(int32_t());
        case GLC_U32: return f(uint32_t());
        case GLC_I64: return f(int64_t());
        case GLC_U64: return f(uint64_t());
        default: return fail(GLC_ERR_INVALID_ARG, "bad dtype");
    }
}

inline unsigned grid_for(int64_t work, int64_t per_block, int64_t cap = 1LL << 30) {
    int64_t g = (work + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return static_cast<unsigned>(g);
}

}  // namespace

template <class T, int FORM>
int launch_fit_t(const void* d_values, glc_column* c, int32_t bs, int32_t fixed_size, hipStream_t s) {
    const T* v = static_cast<const T*>(d_values);
    const FitOut o{c->d_type, c->d_params, c->d_bits, c->d_err};
    const dim3 per_wave(static_cast<unsigned>((c->P + kFitWaves - 1) / kFitWaves));
    const dim3 per_block(static_cast<unsigned>(c->P));
    const int32_t S = fixed_size;
    if (bs != kFitWaveBs) {
        // mixed sizes: a partition a workgroup, as the long ones need; fixed: a wave each
        const int chunk = S > 0 ? kFitWaves : 1;
        hipLaunchKernelGGL((k_fit_any<T, FORM>), dim3(static_cast<unsigned>((c->P + chunk - 1) / chunk)),
                           dim3(64 * kFitWaves), 0, s, v, c->d_start, c->d_end, o, c->P, bs, chunk);
    } else if (S <= 0) {
        // about 8192 workgroups, a chunk of 16 at most (k_fit_chunk's note)
        const int64_t per = (c->P + 8191) / 8192;
        const int chunk = static_cast<int>(per < 1 ? 1 : per > 16 ? 16 : per);
        const int64_t avg = c->n / c->P;
        const dim3 g(static_cast<unsigned>((c->P + chunk - 1) / chunk));
        if (sizeof(T) == 8 && avg > 1024 && avg <= 8192)
            hipLaunchKernelGGL((k_fit_chunk<T, FORM, 3>), g, dim3(256), 0, s, v, c->d_start, c->d_end, o, c->P, chunk);
        else
            hipLaunchKernelGGL((k_fit_chunk<T, FORM, 4>), g, dim3(256), 0, s, v, c->d_start, c->d_end, o, c->P, chunk);
    } else if (S <= 1024) {
        hipLaunchKernelGGL((k_fit_waves<T, FORM, 2>), per_wave, dim3(64 * kFitWaves), 0, s, v, c->d_start, c->d_end, o,
                           c->P);
    } else if (S < kFitWaveMax) {
        hipLaunchKernelGGL((k_fit_waves<T, FORM, 4>), per_wave, dim3(64 * kFitWaves), 0, s, v, c->d_start, c->d_end, o,
                           c->P);
    } else if (S <= kFitRegMax / 2) {
        hipLaunchKernelGGL((k_fit_block<T, FORM, 16>), per_block, dim3(256), 0, s, v, c->d_start, c->d_end, o, c->P);
    } else if (S <= kFitRegMax) {
        hipLaunchKernelGGL((k_fit_block<T, FORM, 32>), per_block, dim3(256), 0, s, v, c->d_start, c->d_end, o, c->P);
    } else {
        hipLaunchKernelGGL((k_fit_block<T, FORM, 0>), per_block, dim3(256), 0, s, v, c->d_start, c->d_end, o, c->P);
    }
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

int launch_fit(int dtype, const void* d_values, glc_column* c, int32_t bs, int fit_form, int32_t fixed_size,
               hipStream_t s) {
    if (c->P == 0) return GLC_OK;
    if (bs < 32 || bs > kFitWaveBs) return fail(GLC_ERR_INVALID_ARG, "fit block size out of range");
    if (fit_form != 0 && fit_form != 1) return fail(GLC_ERR_INVALID_ARG, "fit_form must be 0 or 1");
    return dispatch_dtype(dtype, [&](auto t) {
        using T = decltype(t);
        return fit_form == 0 ? launch_fit_t<T, 0>(d_values, c, bs, fixed_size, s)
                             : launch_fit_t<T, 1>(d_values, c, bs, fixed_size, s);
    });
}

// Offsets (scan: from the widths, else those in the arena), decode index and
// summary; *small: the tile records are built too (launch_build_tinfo otherwise,
// once the summary has been checked).
int launch_index(glc_column* c, bool scan, IndexSummary* d_sum, IndexSummary* h_sum, bool* small, hipStream_t s) {
    *small = false;
    if (c->P == 0) return GLC_OK;
    const IndexIn a{c->d_start, c->d_end, c->d_type, c->d_params, c->d_bits, c->P,
                    c->n,       c->n_index, c->d_desc, c->d_tile_part};
    if (c->P <= kIndexSmall && c->n_index - 1 <= kIndexSmall) {
        *small = true;
        if (scan)
            hipLaunchKernelGGL(k_index_small<true>, dim3(1), dim3(kIndexThreads), 0, s, a, c->d_off, c->d_tinfo, d_sum,
                               h_sum);
        else
            hipLaunchKernelGGL(k_index_small<false>, dim3(1), dim3(kIndexThreads), 0, s, a, c->d_off, c->d_tinfo, d_sum,
                               h_sum);
        GLC_HIP(hipGetLastError());
        return GLC_OK;
    }
    if (scan) {
        int64_t* d_total = reinterpret_cast<int64_t*>(d_sum) + 8;  // scratch slot after the summary
        const int rc = launch_scan(LenBits{c->d_start, c->d_end, c->d_bits}, c->P, c->d_off, d_total, s);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_build_index, dim3(grid_for(c->P, kIndexThreads)), dim3(kIndexThreads), 0, s, a, c->d_off, d_sum,
                       h_sum);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

// Before a column's kernels, instead of clearing the whole arena: the
// partitions (fixed: [pS, min((p+1)S, n)); else copied from src_st / src_en, or
// already there when those are null), the initial model type (host PartitionInfo
// init, G:409-414), for lists that may hold empty partitions (which the fit
// skips) zero outputs, and the summary.
__global__ void k_column_setup(int32_t* __restrict__ st, int32_t* __restrict__ en, int32_t* __restrict__ type,
                               double* __restrict__ params, int32_t* __restrict__ bits, int64_t* __restrict__ err,
                               int64_t P, int64_t n, int32_t S, const int32_t* __restrict__ src_st,
                               const int32_t* __restrict__ src_en, bool empties,
                               IndexSummary* __restrict__ sum) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p == 0) *sum = IndexSummary{};
    if (p >= P) return;
    if (S > 0) {
        const int64_t s0 = p * S;
        st[p] = static_cast<int32_t>(s0);
        en[p] = static_cast<int32_t>(s0 + S < n ? s0 + S : n);
    } else if (src_st) {
        st[p] = src_st[p];
        en[p] = src_en[p];
    }
    type[p] = MODEL_LINEAR;
    if (empties) {
        params[4 * p] = 0.0; params[4 * p + 1] = 0.0; params[4 * p + 2] = 0.0; params[4 * p + 3] = 0.0;
        bits[p] = 0;
        err[p] = 0;
    }
}

int launch_column_setup(glc_column* c, int32_t S, const int32_t* src_st, const int32_t* src_en, bool empties,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_column_setup, dim3(grid_for(c->P, 256)), dim3(256), 0, s, c->d_start, c->d_end,
                       c->d_type, c->d_params, c->d_bits, c->d_err, c->P, c->n, S, src_st, src_en, empties,
                       summary_ptr(c));
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

int launch_build_tinfo(glc_column* c, hipStream_t s) {
    const int64_t ntiles = c->n_index - 1;
    if (c->P == 0 || ntiles <= 0) return GLC_OK;
    hipLaunchKernelGGL(k_build_tinfo, dim3(grid_for(ntiles, 256)), dim3(256), 0, s, c->d_desc, c->d_tile_part, c->n,
                       c->d_tinfo, ntiles);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

// Columns with partition-spanning tiles: tile t's first payload word and the
// three words ending at the one past its last element's first bit hold every
// word that the pack kernels write with atomicOr (the edges of merge_edges and
// merge_span_edges); every other word of the payload is stored whole, so these
// are all a compress must clear.  (2^28 uint64 V6: 19 us, now not run.)
__global__ void k_zero_edges(const Desc* __restrict__ desc, const int32_t* __restrict__ tile_part, int64_t n,
                             int64_t ntiles, uint32_t* __restrict__ words) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    const int64_t e0 = t * kIndexTile;
    const int64_t e1 = (e0 + kIndexTile < n) ? e0 + kIndexTile : n;
    const int64_t plo = tile_part[e0 >> kIndexShift];
    const int64_t phi = tile_part[(e1 + kIndexTile - 1) >> kIndexShift];
    const int64_t wbase = bitpos_lb(desc, plo, phi, e0) >> 5;
    const int64_t last = bitpos_lb(desc, plo, phi, e1 - 1);
    const int64_t wlast = (last >= 0) ? (last + 64) >> 5 : wbase;
    words[wbase] = 0u;
    for (int64_t w = (wlast - 2 > wbase) ? wlast - 2 : wbase + 1; w <= wlast; ++w) words[w] = 0u;
}

int launch_zero_edges(glc_column* c, hipStream_t s) {
    const int64_t ntiles = c->n_index - 1;
    if (c->P == 0 || c->n == 0 || c->total_bits == 0 || ntiles <= 0 || !c->spans) return GLC_OK;
    hipLaunchKernelGGL(k_zero_edges, dim3(grid_for(ntiles, 256)), dim3(256), 0, s, c->d_desc, c->d_tile_part, c->n,
                       ntiles, c->d_words);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

int launch_pack(int dtype, const void* d_values, glc_column* c, hipStream_t s) {
    if (c->P == 0 || c->n == 0 || c->total_bits == 0) return GLC_OK;
    return dispatch_dtype(dtype, [&](auto t) {
        using T = decltype(t);
        const int64_t ntiles = c->n_index - 1;
        if (!c->spans) {
            hipLaunchKernelGGL((k_pack_wave<T, false>), dim3(grid_for(ntiles, kPackWaves)), dim3(64 * kPackWaves), 0, s,
                               static_cast<const T*>(d_values), c->d_desc, c->d_tinfo, c->n, c->d_words);
            GLC_HIP(hipGetLastError());
        } else {
            hipLaunchKernelGGL((k_pack_wave<T, true>), dim3(grid_for(ntiles, kPackWaves)), dim3(64 * kPackWaves), 0, s,
                               static_cast<const T*>(d_values), c->d_desc, c->d_tinfo, c->n, c->d_words);
            GLC_HIP(hipGetLastError());
            // the other tiles, after every wave-packed word
            hipLaunchKernelGGL(k_pack_span<T>, dim3(grid_for(ntiles, kPackWaves)), dim3(64 * kPackWaves), 0, s,
                               static_cast<const T*>(d_values), c->d_desc, c->d_tile_part, c->d_tinfo, c->n,
                               c->d_words);
            GLC_HIP(hipGetLastError());
        }
        return GLC_OK;
    });
}

int v6_capacity(int64_t n, int32_t base, int64_t* cap, int64_t* nvb) {
    if (base < 2 || (base & 1)) return fail(GLC_ERR_INVALID_ARG, "V6 base size must be even and >= 2");
    const int64_t vbs = 8LL * base;
    *nvb = (n + vbs - 1) / vbs;
    *cap = *nvb * ((vbs + base / 2 - 1) / (base / 2));  // at most 16 partitions per variance block
    return GLC_OK;
}

int launch_v6(int dtype, const void* d_values, int64_t n, int32_t base, int32_t* d_start, int32_t* d_end,
              int64_t cap, int64_t* d_total, int64_t* d_base, float* d_var, float* d_thr, int64_t* h_out, hipStream_t s) {
    int64_t need = 0, nvb = 0;
    int rc = v6_capacity(n, base, &need, &nvb);
    if (rc) return rc;
    if (cap < need) return fail(GLC_ERR_INVALID_ARG, "V6 partition buffer too small");
    const int64_t vbs = 8LL * base;
    rc = dispatch_dtype(dtype, [&](auto t) {
        using T = decltype(t);
        const unsigned g = static_cast<unsigned>(nvb < (1LL << 30) ? nvb : (1LL << 30));
        hipLaunchKernelGGL(k_v6_var<T>, dim3(g), dim3(kV6Threads), 0, s, static_cast<const T*>(d_values), n, vbs,
                           nvb, d_var);
        GLC_HIP(hipGetLastError());
        return GLC_OK;
    });
    if (rc) return rc;
    const V6Count f{d_var, d_thr, vbs, n, base};
    if (nvb <= kV6Small) {
        hipLaunchKernelGGL(k_v6_small, dim3(1), dim3(1024), 0, s, f, nvb, d_start, d_end, d_total, h_out);
        GLC_HIP(hipGetLastError());
        return GLC_OK;
    }
    hipLaunchKernelGGL(k_v6_select, dim3(1), dim3(1024), 0, s, d_var, nvb, d_thr);
    GLC_HIP(hipGetLastError());
    rc = launch_scan(f, nvb, d_base, d_total, s);  // per-block partition bases, P
    if (rc) return rc;
    hipLaunchKernelGGL(k_v6_emit, dim3(grid_for(nvb, 256)), dim3(256), 0, s, f, nvb, d_base, d_start, d_end, d_total,
                       h_out);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

__global__ void k_fixed_parts_batch(const BatchCol* __restrict__ cols, const int32_t* __restrict__ part_col,
                                    int64_t Ptot, int32_t S) {
    const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= Ptot) return;
    const BatchCol& c = cols[part_col[g]];
    const int64_t p = g - c.part_base;
    const int64_t s0 = p * S;
    c.start[p] = static_cast<int32_t>(s0);
    c.end[p] = static_cast<int32_t>((s0 + S < c.n) ? s0 + S : c.n);
    c.type[p] = MODEL_LINEAR;  // host PartitionInfo init, G:409-414
}

__global__ void k_batch_prologue(const BatchCol* __restrict__ cols, int C) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < C) *cols[i].sum = IndexSummary{};
}

// Zero the payload words a 1024-element tile can share with its neighbours
// (its first word and last three, which hold every word the pack kernels OR
// into); every other payload word is written whole by exactly one tile.
__global__ void k_zero_edges_batch(const BatchCol* __restrict__ cols, const int32_t* __restrict__ tile_col,
                                   int64_t Ttot) {
    const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= Ttot) return;
    const BatchCol& c = cols[tile_col[g]];
    if (c.payload_words > c.words_reserved) return;
    const int64_t t = g - c.tile_base;
    const int64_t e0 = t * kIndexTile;
    const int64_t e1 = (e0 + kIndexTile < c.n) ? e0 + kIndexTile : c.n;
    const int64_t plo = c.tile_part[e0 >> kIndexShift];
    const int64_t phi = c.tile_part[(e1 + kIndexTile - 1) >> kIndexShift];
    const int64_t wbase = bitpos_lb(c.desc, plo, phi, e0) >> 5;
    const int64_t last = bitpos_lb(c.desc, plo, phi, e1 - 1);
    const int64_t wlast = (last >= 0) ? (last + 64) >> 5 : wbase;
    c.words[wbase] = 0u;
    for (int64_t w = (wlast - 2 > wbase) ? wlast - 2 : wbase + 1; w <= wlast; ++w) c.words[w] = 0u;
}

__global__ void k_set_payload_words(BatchCol* __restrict__ cols, const int64_t* __restrict__ col_bits, int C) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    const int64_t w = (col_bits[i] + 31) / 32;
    cols[i].payload_words = w;
    if (w > cols[i].words_reserved) cols[i].sum->bad_bits = 1;  // cannot happen: reserve is the worst case
}

int launch_batch_compress(const BatchPlan& b, hipStream_t s) {
    if (b.Ptot == 0) return GLC_OK;
    const bool small = b.Pmax <= kBatchSmall && b.Tmax <= kBatchSmall;
    if (!small) {
        hipLaunchKernelGGL(k_batch_prologue, dim3(grid_for(b.C, 256)), dim3(256), 0, s, b.cols, b.C);
        GLC_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_fixed_parts_batch, dim3(grid_for(b.Ptot, 256)), dim3(256), 0, s, b.cols, b.part_col, b.Ptot,
                       b.S);
    GLC_HIP(hipGetLastError());
    const dim3 gf(static_cast<unsigned>((b.Ptot + kFitWaves - 1) / kFitWaves));
    if (b.S <= 1024)
        hipLaunchKernelGGL(k_fit_wave_batch<1024>, gf, dim3(64 * kFitWaves), 0, s, b.cols, b.part_col, b.Ptot, b.S);
    else if (b.S <= kFitWaveMax)
        hipLaunchKernelGGL(k_fit_wave_batch<2048>, gf, dim3(64 * kFitWaves), 0, s, b.cols, b.part_col, b.Ptot, b.S);
    else
        hipLaunchKernelGGL(k_fit_wave_batch<0>, gf, dim3(64 * kFitWaves), 0, s, b.cols, b.part_col, b.Ptot, b.S);
    GLC_HIP(hipGetLastError());
    if (small) {
        hipLaunchKernelGGL(k_batch_index, dim3(static_cast<unsigned>(b.C)), dim3(kBatchIndexThreads), 0, s, b.cols,
                           b.col_bits);
        GLC_HIP(hipGetLastError());
    } else {
        hipLaunchKernelGGL(k_scan_batch, dim3(static_cast<unsigned>(b.C)), dim3(kScanThreads), 0, s, b.cols,
                           b.col_bits);
        GLC_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_build_index_batch, dim3(grid_for(b.Ptot, 256)), dim3(256), 0, s, b.cols, b.part_col,
                           b.Ptot);
        GLC_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_build_tinfo_batch, dim3(grid_for(b.Ttot, 256)), dim3(256), 0, s, b.cols, b.tile_col,
                           b.Ttot);
        GLC_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_set_payload_words, dim3(grid_for(b.C, 256)), dim3(256), 0, s, b.cols, b.col_bits,
                           b.C);
        GLC_HIP(hipGetLastError());
    }
    const unsigned gp = grid_for(b.Ttot, kPackWaves);
    if (b.S % kIndexTile == 0) {  // no tile spans partitions
        hipLaunchKernelGGL(k_pack_wave_batch<false>, dim3(gp), dim3(64 * kPackWaves), 0, s, b.cols, b.tile_col, b.Ttot);
        GLC_HIP(hipGetLastError());
        return GLC_OK;
    }
    hipLaunchKernelGGL(k_zero_edges_batch, dim3(grid_for(b.Ttot, 256)), dim3(256), 0, s, b.cols, b.tile_col, b.Ttot);
    GLC_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_pack_wave_batch<true>, dim3(gp), dim3(64 * kPackWaves), 0, s, b.cols, b.tile_col, b.Ttot);
    GLC_HIP(hipGetLastError());
    // the partition-spanning tiles, after every wave-packed word
    hipLaunchKernelGGL(k_pack_span_batch, dim3(gp), dim3(64 * kPackWaves), 0, s, b.cols, b.tile_col, b.Ttot);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

int launch_fill_u32(uint32_t* p, int64_t n, uint32_t v, hipStream_t s) {
    if (n <= 0) return GLC_OK;
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256, 4096)), dim3(256), 0, s, p, n, v);
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

}  // namespace glc
