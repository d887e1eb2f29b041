// glc_splitmerge.hip -- GPU split/merge partitioner (GLC_PART_GPU_SPLITMERGE).
//
// Algorithm of the reference's VariableLengthPartitioner
// (compression/CpuPartitioner.cuh:141-242) with its cost model (:78-138:
// 80 B + n*bits/8, linear fit without FMA, the int32 n*(n-1) of :56-72), the
// normal-equation sums Sy, Sxy taken exactly in 128-bit integers and rounded
// once to double.  Exact sums are independent of summation order, so the
// parallel reductions here give the same costs -- hence the same boundaries --
// as a sequential evaluation of the same definition.
//
//   blocks  the column is cut into blocks of B values (B divides m, at most
//           128).  Per block: exact sums (prefix sums over the column, so any
//           candidate's sums are two differences) and the vertices of the convex
//           hull of its points (k_sm_blocks), about 11 for 128 noisy values;
//   split   every start s = j*m (m = minimum size) is evaluated at once: the
//           candidate sizes m*{1,2,3,4,5,7,...,17,21,25,29} (step m, then 2m
//           above 4m, then 4m above 16m, at most 32m); the smallest cost per
//           value wins (first on ties);
//   chain   the greedy walk 0 -> end(0) -> end(end(0)) ... keeps the starts it
//           reaches: pointer doubling inside chunks, one walk over the chunks;
//   merge   up to 10 left-to-right passes.  The group that starts at a
//           partition does not depend on how the walk got there, so every
//           partition's group is grown at once, one wave each (k_sm_grow), and
//           the chain keeps the groups the walk from partition 0 reaches.  A
//           wave grows its group for a bounded number of steps; the groups that
//           want more are grown on, one after the other, where the walk reaches
//           them (k_sm_more, k_sm_walk).
//
// The maximum residual of a line over a range.  A cost needs only the bit
// width of max |v_i - round(pr_i)|, pr_i = t0 + t1 * i in FP64.  Over a block the
// real-valued residual of any line is largest at a hull vertex, so with D the
// largest |v - pr| and H the largest |v - round(pr)| over the vertices,
//     max(H, D - f) <= max <= D + f,  f = 0.5 + 4 eps + 2^-50 D,
//     eps = 2^-52 (|t0| + |t1| n)
// (one prediction's FP64 error is at most eps; D's own, each vertex as one fused
// y - t1 x less the block's t0 + t1 x0, at most eps + 2^-52 D; values and
// predictions within 2^52, where every difference of two integers is exact).  D
// alone first; H, at more than twice the instructions a vertex, only where a power
// of two lies between its bounds.  Both ends then have the same bit width except
// where one lies between these too; there, and for blocks or candidates outside
// the exact range, the values themselves are read.  That makes one evaluation about 10 times cheaper than a pass over the values: 2^26 uint64
// piecewise-linear values, m = 128: split 8.1 -> 0.73 ms (1.13 with D and H at
// once), and growing every partition's group takes 0.28 ms a pass where the
// sequential walk (one workgroup regrowing groups across segments) took 23.4 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <map>
#include <mutex>
#include <vector>

#include "glc_device.hpp"
#include "glc_internal.hpp"

namespace glc {
namespace {

constexpr int kSmThreads = 256;
constexpr int kPfxChunk = 64;  // block-prefix positions per chunk (k_sm_blocks, k_sm_chunk_pfx)
constexpr int kMaxCand = 14;  // m * {1,2,3,4,5,7,9,11,13,15,17,21,25,29}
__constant__ int kCandUnits[kMaxCand] = {1, 2, 3, 4, 5, 7, 9, 11, 13, 15, 17, 21, 25, 29};
// units of the candidates before candidate k (of one start)
__constant__ int kCandCum[kMaxCand + 1] = {0, 1, 3, 6, 10, 15, 22, 31, 42, 55, 70, 87, 108, 133, 162};

typedef __int128 i128;
typedef unsigned __int128 u128;

template <class T> __device__ __forceinline__ i128 wide(T x) {
    if constexpr (std::is_signed<T>::value) return static_cast<i128>(static_cast<int64_t>(x));
    else return static_cast<i128>(static_cast<uint64_t>(x));
}

// Round-to-nearest-even conversion of a signed 128-bit integer to double.
__device__ double i128_to_double(i128 x) {
    const bool neg = x < 0;
    const u128 m = neg ? static_cast<u128>(0) - static_cast<u128>(x) : static_cast<u128>(x);
    const uint64_t hi = static_cast<uint64_t>(m >> 64), lo = static_cast<uint64_t>(m);
    if (hi == 0 && lo == 0) return 0.0;
    const int L = hi ? 127 - __builtin_clzll(hi) : 63 - __builtin_clzll(lo);
    double r;
    if (L <= 52) {
        r = static_cast<double>(lo);
    } else {
        const int sh = L - 52;
        uint64_t mant = static_cast<uint64_t>(m >> sh);
        const u128 rem = m & ((static_cast<u128>(1) << sh) - 1);
        const u128 half = static_cast<u128>(1) << (sh - 1);
        if (rem > half || (rem == half && (mant & 1))) ++mant;
        r = __builtin_ldexp(static_cast<double>(mant), sh);  // mant <= 2^53: exact
    }
    return neg ? -r : r;
}

__device__ __forceinline__ i128 shfl_xor_i128(i128 v, int o) {
    const uint64_t lo = static_cast<uint64_t>(static_cast<u128>(v));
    const uint64_t hi = static_cast<uint64_t>(static_cast<u128>(v) >> 64);
    const uint64_t l2 = __shfl_xor(lo, o, 64), h2 = __shfl_xor(hi, o, 64);
    return static_cast<i128>((static_cast<u128>(h2) << 64) | l2);
}
__device__ __forceinline__ i128 wave_sum(i128 v) {
    for (int o = 32; o > 0; o >>= 1) v += shfl_xor_i128(v, o);
    return v;
}
__device__ __forceinline__ int64_t wave_max(int64_t v) {
    for (int o = 32; o > 0; o >>= 1) {
        const int64_t y = __shfl_xor(v, o, 64);
        v = y > v ? y : v;
    }
    return v;
}

// sum of i^2 for i < n, (n-1) n (2n-1) / 6, for 1 <= n < 2^31 without a
// 128-bit division: one of n-1, n is even and one of n-1, n, 2n-1 is a
// multiple of 3, so the division is exact on the factors.
__device__ __forceinline__ i128 sum_sq(int64_t n) {
    uint64_t a = static_cast<uint64_t>(n - 1), b = static_cast<uint64_t>(n), c = static_cast<uint64_t>(2 * n - 1);
    if (a % 2 == 0) a /= 2;
    else b /= 2;
    if (a % 3 == 0) a /= 3;
    else if (b % 3 == 0) b /= 3;
    else c /= 3;
    return static_cast<i128>(static_cast<u128>(a * b) * c);  // a * b < 2^62, c < 2^32
}

// theta of the split/merge cost model from exact sums over n values.
__device__ void sm_theta(i128 Sy, i128 Sxy, int64_t n, double& t0, double& t1) {
    const i128 Sxx = sum_sq(n);
    const int32_t nn1 = static_cast<int32_t>(static_cast<uint32_t>(n) * static_cast<uint32_t>(n - 1));
    const double sx = static_cast<double>(nn1) / 2.0;
    const double sy = i128_to_double(Sy), sxy = i128_to_double(Sxy), sxx = i128_to_double(Sxx);
    const double dn = static_cast<double>(n);
    const double det = dn * sxx - sx * sx;
    if (__builtin_fabs(det) > 1e-10) {
        t1 = (dn * sxy - sx * sy) / det;
        t0 = (sy - t1 * sx) / dn;
    } else {
        t1 = 0.0;
        t0 = sy / dn;
    }
}

template <class T> __device__ __forceinline__ int64_t abs_err(T v, double t0, double t1, int64_t i) {
    const double pr = t0 + t1 * static_cast<double>(i);  // no contraction (-ffp-contract=off)
    const int64_t d = calc_delta<T>(v, x86_cast<T>(round_away(pr)));  // the host cost model's conversion
    return d < 0 ? static_cast<int64_t>(0ULL - static_cast<uint64_t>(d)) : d;
}

// Residual magnitude in FP64 when it is exact.  For values v and rounded
// predictions p of magnitude <= 2^52 (inside T for 32-bit types), x86_cast is
// the identity on p, calc_delta is v - p without wrap or saturation, and the
// FP64 difference of two such integers is exact; so fabs(v - round(pr)) is
// abs_err's result.  The prediction t0 + t1 * i is monotonic in i, so its two
// end values bound a candidate's whole range.
constexpr double kExact = 4503599627370496.0;  // 2^52
template <class T> __device__ __forceinline__ bool small_value(T x) {
    if constexpr (sizeof(T) == 4) return true;
    else if constexpr (std::is_signed<T>::value) return x >= -(int64_t(1) << 52) && x <= (int64_t(1) << 52);
    else return x <= (uint64_t(1) << 52);
}
template <class T> __device__ __forceinline__ bool small_pred(double pr) {  // false for NaN
    if constexpr (std::is_same<T, int32_t>::value) return pr >= -2147483647.0 && pr <= 2147483646.0;
    else if constexpr (std::is_same<T, uint32_t>::value) return pr >= 0.0 && pr <= 4294967294.0;
    else if constexpr (std::is_signed<T>::value) return pr >= -kExact && pr <= kExact;
    else return pr >= 0.0 && pr <= kExact;
}

__device__ __forceinline__ int32_t bits_of(int64_t mx) {
    if (mx <= 0) return 0;
    const int b = 64 - __builtin_clzll(static_cast<unsigned long long>(mx)) + 1;
    return b > 64 ? 64 : b;
}

__device__ __forceinline__ double cost_of(int64_t n, int32_t bits) {
    return 80.0 + static_cast<double>(n) * bits / 8.0;  // CpuPartitioner.cuh:128-138
}

template <int NT> struct FitLdsT {
    i128 sy[NT / 64];
    i128 sxy[NT / 64];
    int64_t mx[NT / 64];
    double t0, t1, cost;
    int fast;  // both end predictions within small_pred's range
};
typedef FitLdsT<kSmThreads> FitLds;

// Prefix sums of the column at block granularity: G1(p) = sum of y_q and
// G2(p) = sum of q * y_q over q < min(p * B, n), for p in [0, JB].
// G(p) = p(p) + c(p / kPfxChunk).
struct SmPrefix {
    const i128 *p1, *p2, *c1, *c2;
    int64_t n, JB;
    int32_t B;
};
__device__ __forceinline__ i128 pfx_at(const i128* p, const i128* c, int64_t i) {
    return p[i] + c[i / kPfxChunk];
}

// the block that starts at position s (s < 2^31: 32-bit division)
__device__ __forceinline__ int64_t block_of(const SmPrefix& pf, int64_t s) {
    return static_cast<uint32_t>(s) / static_cast<uint32_t>(pf.B);
}

// Hull vertices of the blocks: vertex k of block b at
// ((b / 64) * slots + k) * 64 + b % 64, so that lanes on consecutive blocks read
// consecutive memory; y its value, x its index in the block.  nv[b]: the number of
// vertices, or kHullScan for a block that has to be read value by value (more
// than `slots` vertices, or a value outside small_value's range).  slots = 0: no
// hulls, every range is read.
constexpr int kHullSlots = 24;
constexpr int kHullScan = 255;
constexpr int kHullMaxB = 128;
struct SmHull {
    double* y;
    uint8_t* x;
    uint8_t* nv;
    int32_t slots;
};
__device__ __forceinline__ int64_t hull_at(int32_t slots, int64_t b, int k) {
    return ((b >> 6) * slots + k) * 64 + (b & 63);
}

// A candidate's line over [s, e) (s a block start, e one or n) from the
// prefix sums, and whether its two end predictions are within small_pred.
template <class T>
__device__ __forceinline__ void range_line(const SmPrefix& pf, int64_t s, int64_t e, double& t0, double& t1,
                                           bool& fast) {
    const int64_t ib = block_of(pf, s), ie = (e == pf.n) ? pf.JB : block_of(pf, e);
    const i128 sy = pfx_at(pf.p1, pf.c1, ie) - pfx_at(pf.p1, pf.c1, ib);
    const i128 sxy = pfx_at(pf.p2, pf.c2, ie) - pfx_at(pf.p2, pf.c2, ib) - static_cast<i128>(s) * sy;
    sm_theta(sy, sxy, e - s, t0, t1);
    fast = small_pred<T>(t0 + t1 * 0.0) && small_pred<T>(t0 + t1 * static_cast<double>(e - s - 1));
}

// Largest residual magnitude of values x0, x0 + step, ... < n of a range at v
// (four loads in flight; one lane's share).
template <class T>
__device__ __forceinline__ int64_t scan_err(const T* __restrict__ v, int64_t x0, int64_t n, int step, double t0,
                                            double t1, bool fast) {
    int64_t mx = 0;
    double md = 0.0;
    for (int64_t i0 = x0; i0 < n; i0 += 4 * step) {
        T x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {  // index clamped; the extra ones are skipped
            const int64_t i = i0 + k * step;
            x[k] = v[i < n ? i : n - 1];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t i = i0 + k * step;
            if (i >= n) break;
            if (fast && small_value<T>(x[k])) {
                const double pr = t0 + t1 * static_cast<double>(i);  // no contraction (-ffp-contract=off)
                md = __builtin_fmax(md, __builtin_fabs(static_cast<double>(x[k]) - round_away(pr)));
            } else {
                const int64_t a = abs_err<T>(x[k], t0, t1, i);
                mx = a > mx ? a : mx;
            }
        }
    }
    const int64_t mdi = static_cast<int64_t>(md);
    return mdi > mx ? mdi : mx;
}

// D (see the top of the file) over the vertices of one block whose first value
// has index x0 in the range.  y, x: the block's vertices, `stride` apart.
__device__ __forceinline__ double hull_far(const double* __restrict__ y, const uint8_t* __restrict__ x, int stride,
                                           int nv, int32_t x0, double t0, double t1) {
    double hi = -DBL_MAX, lo = DBL_MAX;
#pragma unroll 4
    for (int k = 0; k < nv; ++k) {
        const double r = __builtin_fma(-t1, static_cast<double>(x[k * stride]), y[k * stride]);
        hi = __builtin_fmax(hi, r);
        lo = __builtin_fmin(lo, r);
    }
    const double base = __builtin_fma(t1, static_cast<double>(x0), t0);
    return __builtin_fmax(hi - base, base - lo);
}

// H over the same.
__device__ __forceinline__ double hull_low(const double* __restrict__ y, const uint8_t* __restrict__ x, int stride,
                                           int nv, int32_t x0, double t0, double t1) {
    double H = 0.0;
    for (int k = 0; k < nv; ++k) {
        const double pr = t0 + t1 * static_cast<double>(x0 + x[k * stride]);  // no contraction (-ffp-contract=off)
        H = __builtin_fmax(H, __builtin_fabs(y[k * stride] - round_away(pr)));
    }
    return H;
}

// The bit width that D and H (both <= 2^53 + 1) settle for a range of n
// values, -1 if a power of two lies between the two bounds.  H = 0: from D
// alone.
__device__ __forceinline__ int32_t hull_bits(double D, double H, double t0, double t1, int64_t n) {
    const double eps = (__builtin_fabs(t0) + __builtin_fabs(t1) * static_cast<double>(n)) * 0x1p-52;
    const double far = D * 0x1p-50 + 0.5 + 4.0 * eps;
    const int32_t lo = bits_of(static_cast<int64_t>(__builtin_ceil(__builtin_fmax(H, D - far))));
    const int32_t hi = bits_of(static_cast<int64_t>(D + far));
    return lo == hi ? lo : -1;
}

// Cost of [s, e) by a pass for the sums and one for the maximum residual,
// computed by the whole workgroup (all threads call it).
template <class T, int NT = kSmThreads>
__device__ double wg_cost(const T* __restrict__ v, int64_t s, int64_t e, FitLdsT<NT>& L) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t n = e - s;
    i128 sy = 0, sxy = 0;
    for (int64_t i = tid; i < n; i += NT) {
        const i128 y = wide<T>(v[s + i]);
        sy += y;
        sxy += y * static_cast<i128>(i);
    }
    sy = wave_sum(sy);
    sxy = wave_sum(sxy);
    if (lane == 0) {
        L.sy[w] = sy;
        L.sxy[w] = sxy;
    }
    __syncthreads();
    if (tid == 0) {
        i128 a = 0, b = 0;
#pragma unroll 1
        for (int k = 0; k < NT / 64; ++k) {
            a += L.sy[k];
            b += L.sxy[k];
        }
        sm_theta(a, b, n, L.t0, L.t1);
        L.fast = small_pred<T>(L.t0 + L.t1 * 0.0) && small_pred<T>(L.t0 + L.t1 * static_cast<double>(n - 1));
    }
    __syncthreads();
    const int64_t mx = wave_max(scan_err<T>(v + s, tid, n, NT, L.t0, L.t1, L.fast != 0));
    if (lane == 0) L.mx[w] = mx;
    __syncthreads();
    if (tid == 0) {
        int64_t m = L.mx[0];
#pragma unroll 1
        for (int k = 1; k < NT / 64; ++k) m = L.mx[k] > m ? L.mx[k] : m;
        L.cost = cost_of(n, bits_of(m));
    }
    __syncthreads();
    const double c = L.cost;
    __syncthreads();  // L is reused by the caller's next fit
    return c;
}

// ---- split: one workgroup per start j*m ------------------------------------
template <class T>
__global__ __launch_bounds__(kSmThreads) void k_sm_split(const T* __restrict__ v, int64_t n, int32_t m, int64_t J,
                                                         int32_t* __restrict__ best_end,
                                                         double* __restrict__ best_cost) {
    __shared__ i128 s_seg[kMaxCand][2];
    __shared__ double s_t[kMaxCand][2];
    __shared__ int64_t s_mx[kSmThreads / 64][kMaxCand];
    __shared__ bool s_fast[kMaxCand];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t j = blockIdx.x;
    if (j >= J) return;
    const int64_t cur = j * m;
    const int64_t max_size = (n - cur < static_cast<int64_t>(m) * 32) ? n - cur : static_cast<int64_t>(m) * 32;
    int K = 0;
    while (K < kMaxCand && static_cast<int64_t>(kCandUnits[K]) * m <= max_size) ++K;
    if (K == 0) {  // fewer than m values left: one partition [cur, n)
        __shared__ FitLds L;
        const double c = wg_cost<T>(v, cur, n, L);
        if (tid == 0) {
            best_end[j] = static_cast<int32_t>(n);
            best_cost[j] = c;
        }
        return;
    }
    const int64_t Lmax = static_cast<int64_t>(kCandUnits[K - 1]) * m;
    int big = 0;  // a value outside small_value's range
    // segment sums: segment k = [size(k-1), size(k)), one wave each
    for (int k = w; k < K; k += kSmThreads / 64) {
        const int64_t a = (k == 0) ? 0 : static_cast<int64_t>(kCandUnits[k - 1]) * m;
        const int64_t b = static_cast<int64_t>(kCandUnits[k]) * m;
        i128 sy = 0, sxy = 0;
        for (int64_t i = a + lane; i < b; i += 64) {
            const T x = v[cur + i];
            big |= small_value<T>(x) ? 0 : 1;
            const i128 y = wide<T>(x);
            sy += y;
            sxy += y * static_cast<i128>(i);
        }
        sy = wave_sum(sy);
        sxy = wave_sum(sxy);
        if (lane == 0) {
            s_seg[k][0] = sy;
            s_seg[k][1] = sxy;
        }
    }
    const int any_big = __syncthreads_or(big);
    if (tid < K) {
        i128 sy = 0, sxy = 0;
        for (int k = 0; k <= tid; ++k) {
            sy += s_seg[k][0];
            sxy += s_seg[k][1];
        }
        double t0, t1;
        const int64_t size = static_cast<int64_t>(kCandUnits[tid]) * m;
        sm_theta(sy, sxy, size, t0, t1);
        s_t[tid][0] = t0;
        s_t[tid][1] = t1;
        const double p0 = t0 + t1 * 0.0, p1 = t0 + t1 * static_cast<double>(size - 1);
        s_fast[tid] = small_pred<T>(p0) && small_pred<T>(p1);
    }
    __syncthreads();
    bool fast = !any_big;
    for (int k = 0; k < K; ++k) fast = fast && s_fast[k];
    int64_t mx[kMaxCand];
#pragma unroll
    for (int k = 0; k < kMaxCand; ++k) mx[k] = 0;
    if (fast) {  // every candidate's residuals exact in FP64 (workgroup-uniform)
        double md[kMaxCand];
#pragma unroll
        for (int k = 0; k < kMaxCand; ++k) md[k] = 0.0;
        for (int64_t i = tid; i < Lmax; i += kSmThreads) {
            const double y = static_cast<double>(v[cur + i]);
            const double xi = static_cast<double>(i);
#pragma unroll
            for (int k = 0; k < kMaxCand; ++k) {
                if (k < K && i < static_cast<int64_t>(kCandUnits[k]) * m) {
                    const double pr = s_t[k][0] + s_t[k][1] * xi;  // no contraction (-ffp-contract=off)
                    md[k] = __builtin_fmax(md[k], __builtin_fabs(y - round_away(pr)));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < kMaxCand; ++k) mx[k] = static_cast<int64_t>(md[k]);
    } else {
        for (int64_t i = tid; i < Lmax; i += kSmThreads) {
            const T x = v[cur + i];
#pragma unroll
            for (int k = 0; k < kMaxCand; ++k) {
                if (k < K && i < static_cast<int64_t>(kCandUnits[k]) * m) {
                    const int64_t a = abs_err<T>(x, s_t[k][0], s_t[k][1], i);
                    mx[k] = a > mx[k] ? a : mx[k];
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kMaxCand; ++k) {
        const int64_t r = wave_max(mx[k]);
        if (lane == 0) s_mx[w][k] = r;
    }
    __syncthreads();
    if (tid == 0) {
        double best = DBL_MAX, bc = 0.0;
        int64_t be = (cur + m < n) ? cur + m : n;
        for (int k = 0; k < K; ++k) {
            int64_t r = s_mx[0][k];
            for (int q = 1; q < kSmThreads / 64; ++q) r = s_mx[q][k] > r ? s_mx[q][k] : r;
            const int64_t size = static_cast<int64_t>(kCandUnits[k]) * m;
            const double c = cost_of(size, bits_of(r));
            const double cpe = c / static_cast<double>(size);
            if (cpe < best) {
                best = cpe;
                be = cur + size;
                bc = c;
            }
        }
        best_end[j] = static_cast<int32_t>(be);
        best_cost[j] = bc;
    }
}

// Block sums, prefixes and hulls.  One workgroup per chunk of kPfxChunk = 64
// blocks, staged in LDS (rows of B | 1 values: 64 lanes reading the same index
// of 64 blocks hit different banks).
//   filter  a block per wave, twice 64 values: hull_filter;
//   hull    wave 0 walks the upper hulls, wave 1 the lower ones, a block per
//           lane: hull_chain;
//   sums    waves 2 to 5, four lanes a block; the last wave scans the 64 blocks'.
// p1, p2 receive the exclusive prefix inside the chunk, c1, c2 the chunk's
// totals (k_sm_chunk_scan turns those into chunk offsets).  A block per lane
// with values straight from memory (one cache line per lane and step) read the
// column at 0.55 TB/s.  Bound by latency: the rows of 64 blocks take half of the
// LDS, so only two workgroups share a CU, and the walk keeps one wave of each hull
// busy.  Hence few candidates and few dependent reads a turn for the walk, rows as
// FP64 (nothing converted in a loop), and 16 waves for the other phases: 2^26
// uint64 values 1002 -> 394 us, one workgroup alone 42 -> 26 us (with 4 waves, six
// distances as the filter and a walk in int64 before).
constexpr int kBlkThreads = 1024;
constexpr int kSumWaves = 4;
constexpr int kHullCand = 56;  // candidates of one hull; more: the block is read

// l <= r (UP) or l >= r for certain, for two products of a difference of values
// (whole, <= 2^53) and one of indices (< 2^7).  Below 2^50 both are exact and so
// is the test; above, their error and the test's is less than the margin.
template <bool UP>
__device__ __forceinline__ bool surely_inside(double l, double r) {
    const double margin = (__builtin_fabs(l) + __builtin_fabs(r)) * 0x1p-51;
    return UP ? l < (r + 0.5) - margin : l > (r - 0.5) + margin;
}

template <bool UP>
__device__ __forceinline__ float row16_best(float x) {  // over the 16 lanes of a row
#define GLC_ROW_STEP(ror)                                                                                  \
    {                                                                                                      \
        const float o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), ror, 0xF, 0xF, true)); \
        x = UP ? __builtin_fmaxf(x, o) : __builtin_fminf(x, o);                                            \
    }
    GLC_ROW_STEP(0x128) GLC_ROW_STEP(0x124) GLC_ROW_STEP(0x122) GLC_ROW_STEP(0x121)
#undef GLC_ROW_STEP
    return x;
}

struct Anchor {
    double x, y;
};
constexpr int kAnchors = kHullMaxB / 16 + 2;  // of one hull: a block's ends and one of every 16 indices

// One block's candidates for the upper and lower hull: their indices in order to
// lu and ld, 64 apart, and their numbers; index i in lane i % 64.  A point above
// the line through the block's ends can only be a vertex of the upper hull, one
// below only of the lower, one on it of neither; and none on or inside a chord of
// two others is.  Chords: between the neighbours, and between anchors, which are
// the ends and, of every 16 indices, the point furthest outside the line through
// them (as float: a poor choice keeps more, nothing else).  One test a point, for
// its side.  Of 128 values with noise 10 to 12 are left for each hull; neighbours
// at distances 1, 2, 4, ... 32 without anchors left 25 to 35, tested for both.
// Where the block has a kink, a line through the ends says little (25 to 50
// left, up to 67): then once more, with the point furthest outside the chord of
// the first anchors.
// a: the wave's, [2][kAnchors].
constexpr int kFewCand = 24;
__device__ __forceinline__ void hull_filter(const double* __restrict__ row, int len, int lane, Anchor* a, uint8_t* lu,
                                            uint8_t* ld, uint8_t* nu, uint8_t* nd) {
    const double y0 = row[0], yl = row[len - 1], dy = yl - y0, n1 = static_cast<double>(len - 1);
    const int halves = len > 64 ? 2 : 1, last = 1 + (len + 15) / 16;
    constexpr uint64_t kRow1 = 0x0001000100010001ULL;  // the first lane of each row
    wave_lds_fence();
    if (lane < 2) {
        a[lane * kAnchors] = Anchor{0.0, y0};
        a[lane * kAnchors + last] = Anchor{n1, yl};
    }
    double y[2];
    float ku[2], kd[2];  // how far outside above (> 0), below (< 0); infinite: no longer asked
    bool up[2], dn[2];
    uint64_t mu[2] = {0, 0}, md[2] = {0, 0};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (half == halves) break;
        const int i = half * 64 + lane;
        const bool in = i < len;
        y[half] = row[i];  // past the block: anything
        const double l = (y[half] - y0) * n1, r = dy * static_cast<double>(i);
        up[half] = in & !surely_inside<true>(l, r);
        dn[half] = in & !surely_inside<false>(l, r);
        const float key = static_cast<float>(l - r);
        ku[half] = in ? key : -__builtin_inff();
        kd[half] = in ? key : __builtin_inff();
    }
    for (int pass = 0;; ++pass) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half == halves) break;
            const double x = static_cast<double>(half * 64 + lane);
            const float bu = row16_best<true>(ku[half]), bd = row16_best<false>(kd[half]);
            const uint64_t eu = __ballot((ku[half] > -__builtin_inff()) & (bu == ku[half]));
            const uint64_t ed = __ballot((kd[half] < __builtin_inff()) & (bd == kd[half]));
            // the first of each row; a row without any keeps its anchor
            const uint64_t zu = eu | kRow1 << 15, zd = ed | kRow1 << 15;
            const uint64_t fu = zu & ~(zu - kRow1) & eu, fd = zd & ~(zd - kRow1) & ed;
            const int e = 1 + half * 4 + (lane >> 4);
            if ((fu >> lane) & 1) a[e] = Anchor{x, y[half]};
            if ((fd >> lane) & 1) a[kAnchors + e] = Anchor{x, y[half]};
        }
        wave_lds_fence();
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half == halves) break;
            const int i = half * 64 + lane;
            const double x = static_cast<double>(i);
            const Anchor* t = a + (up[half] ? 0 : kAnchors) + half * 4 + (lane >> 4);
            const Anchor c = t[1], b = t[0], d = t[2];
            const bool before = x <= c.x, after = x >= c.x;
            const double px = before ? b.x : c.x, py = before ? b.y : c.y;
            const double qx = after ? d.x : c.x, qy = after ? d.y : c.y;
            const double l = (y[half] - py) * (qx - px), r = (qy - py) * (x - px);
            const double l1 = 2.0 * y[half], r1 = row[i - 1] + row[i + 1];
            const bool iu = surely_inside<true>(l, r) | (l1 <= r1), id = surely_inside<false>(l, r) | (l1 >= r1);
            // on an uncertain side of the line: in both lists, without a test for the lower
            const bool end = (i == 0) | (i == len - 1);
            const bool u = up[half] & (end | !iu), w = dn[half] & (end | up[half] | !id);
            const float key = static_cast<float>(l - r) * __builtin_amdgcn_rcpf(static_cast<float>(qx - px));
            ku[half] = u ? key : -__builtin_inff();
            kd[half] = w ? key : __builtin_inff();
            mu[half] = __ballot(u | end);
            md[half] = __ballot(w | end);
            up[half] = u;
            dn[half] = w;
        }
        const int cu = __popcll(mu[0]) + __popcll(mu[1]), cd = __popcll(md[0]) + __popcll(md[1]);
        if (pass == 1 || (cu <= kFewCand && cd <= kFewCand)) {
            if (lane == 0) *nu = static_cast<uint8_t>(cu), *nd = static_cast<uint8_t>(cd);
            break;
        }
        wave_lds_fence();
    }
    auto put = [&](const uint64_t (&m)[2], uint8_t* list) {
        int before = 0;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half == halves) break;
            const int k = before + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                                       m[half] >> 32, __builtin_amdgcn_mbcnt_lo(m[half], 0)));
            if (((m[half] >> lane) & 1) && k < kHullCand) list[k * 64] = static_cast<uint8_t>(half * 64 + lane);
            before += __popcll(m[half]);
        }
    };
    put(mu, lu);
    put(md, ld);
}

// One block's upper (UP) or lower hull among the `left` points whose indices are
// list[0], list[64], ..., into the front of the same list; returns their number.
// A vertex is dropped only where it is inside for certain: one kept in vain costs
// time, never the result.
// Lanes walk blocks of their own, so every turn is one straight run, the same for
// a vertex dropped and a point taken (as two branches the compiler nests them, and
// all lanes wait for the one with the most drops at every point).  The last three
// vertices a, b, c, the index of the fourth and the next two points i, j stay in
// registers, and what a turn reads is first used after the next one's test.
template <bool UP>
__device__ __forceinline__ int hull_chain(const double* __restrict__ row, int32_t B, int left, uint8_t* list) {
    auto at = [&](int k) {  // entries past the points hold anything
        const int x = list[(k < kHullCand ? k : kHullCand - 1) * 64];
        return x < B ? x : B - 1;
    };
    if (left == 0) return 0;
    int n = 0, k = 2, xa = 0, xb = 0, xc = 0, xd = 0, xi = at(0), xj = at(1), xn = at(2);
    double ya = 0.0, yb = 0.0, yc = 0.0, yi = row[xi], yj = row[xj], val = yj;
    bool dropped = false;  // val belongs to c, not to j
    do {
        const bool drop = n >= 2 && surely_inside<UP>((ya - yb) * static_cast<double>(xi - xa),
                                                      (yi - ya) * static_cast<double>(xa - xb));
        yc = dropped ? val : yc;
        yj = dropped ? yj : val;
        list[n * 64] = static_cast<uint8_t>(xi);  // of no account if dropped
        val = row[drop ? xd : xn];
        dropped = drop;
        const double ta = ya, tb = yb;
        const int za = xa, zb = xb;
        ya = drop ? yb : yi;
        xa = drop ? xb : xi;
        yb = drop ? yc : ta;
        xb = drop ? xc : za;
        yc = tb;  // a drop's is on its way
        xc = drop ? xd : zb;
        yi = drop ? yi : yj;
        xi = drop ? xi : xj;
        xj = drop ? xj : xn;
        n += drop ? -1 : 1;
        k += drop ? 0 : 1;
        left -= drop ? 0 : 1;
        xd = at(n < 4 ? 0 : n - 4);
        xn = at(k);
    } while (left > 0);
    return n;
}

__device__ __forceinline__ i128 shfl_up_i128(i128 v, int o) {
    const uint64_t lo = static_cast<uint64_t>(static_cast<u128>(v));
    const uint64_t hi = static_cast<uint64_t>(static_cast<u128>(v) >> 64);
    const uint64_t l2 = __shfl_up(lo, o, 64), h2 = __shfl_up(hi, o, 64);
    return static_cast<i128>((static_cast<u128>(h2) << 64) | l2);
}

inline __host__ __device__ int hull_stride(int32_t B) { return B | 1; }
// The filter reads up to index 128 and -1 of a row, whatever its length.
constexpr int kHullPad0 = 2, kHullPad1 = 66;
inline size_t hull_lds(int32_t B) { return static_cast<size_t>(64 * hull_stride(B) + kHullPad0 + kHullPad1) * 8; }

template <class T>
__global__ __launch_bounds__(kBlkThreads) void k_sm_blocks(const T* __restrict__ v, int64_t n, int32_t B, int64_t JB,
                                                          i128* __restrict__ p1, i128* __restrict__ p2,
                                                          i128* __restrict__ c1, i128* __restrict__ c2, SmHull h) {
    extern __shared__ double s_rows[];  // 64 rows between pads
    double* s_v = s_rows + kHullPad0;
    __shared__ uint8_t s_list[2][kHullCand * 64];  // candidate, then vertex k of block b at k * 64 + b
    __shared__ uint8_t s_n[2][64];
    __shared__ i128 s_sum[2][64];
    __shared__ Anchor s_anchor[kBlkThreads / 64][2 * kAnchors];
    __shared__ int32_t s_big[64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stride = hull_stride(B);
    const uint32_t rcp = 0xFFFFFFFFu / static_cast<uint32_t>(B) + 1u;  // i / B, exact for i * B < 2^32
    const int64_t b0 = static_cast<int64_t>(blockIdx.x) * kPfxChunk;
    const int64_t q0 = b0 * B;
    int32_t cnt = 64 * B;  // values of these 64 blocks
    if (q0 + cnt > n) cnt = n > q0 ? static_cast<int32_t>(n - q0) : 0;
    if (tid < 64) s_big[tid] = 0, s_n[0][tid] = s_n[1][tid] = 0;
    __syncthreads();
    for (int32_t i0 = tid; i0 < cnt; i0 += 8 * kBlkThreads) {
        T y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // eight loads in flight (index clamped)
            const int32_t i = i0 + k * kBlkThreads;
            y[k] = v[q0 + (i < cnt ? i : cnt - 1)];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int32_t i = i0 + k * kBlkThreads;
            if (i >= cnt) break;
            const int32_t blk = B == 1 ? i : static_cast<int32_t>(__umulhi(static_cast<uint32_t>(i), rcp));
            s_v[blk * stride + (i - blk * B)] = static_cast<double>(y[k]);
            if (!small_value<T>(y[k])) s_big[blk] = 1;
        }
    }
    __syncthreads();
    for (int b = w; b < 64; b += kBlkThreads / 64) {  // filter: a block per wave
        const int len = cnt - b * B < B ? cnt - b * B : B;
        if (len > 0)
            hull_filter(s_v + b * stride, len, lane, s_anchor[w], s_list[0] + b, s_list[1] + b, &s_n[0][b], &s_n[1][b]);
    }
    __syncthreads();
    const double* row = s_v + lane * stride;
    if (w == 0) {
        if (s_n[0][lane] <= kHullCand)
            s_n[0][lane] = static_cast<uint8_t>(hull_chain<true>(row, B, s_n[0][lane], s_list[0] + lane));
    } else if (w == 1) {
        if (s_n[1][lane] <= kHullCand)
            s_n[1][lane] = static_cast<uint8_t>(hull_chain<false>(row, B, s_n[1][lane], s_list[1] + lane));
    } else if (w < 2 + kSumWaves) {  // 64 / kSumWaves blocks a wave, kSumWaves lanes a block
        const int blk = (w - 2) * (64 / kSumWaves) + lane / kSumWaves, sub = lane % kSumWaves;
        const int len = cnt - blk * B < B ? cnt - blk * B : B;
        const double* r = s_v + blk * stride;
        i128 a1 = 0, a2 = 0;  // sum of y, of i * y
        if (s_big[blk]) {
            for (int i = sub; i < len; i += kSumWaves) {
                const i128 y = wide<T>(v[q0 + static_cast<int64_t>(blk) * B + i]);
                a1 += y;
                a2 += y * static_cast<i128>(i);
            }
        } else {  // |y| <= 2^52: a block's sum fits 64 bits, eight products too
            int64_t s1 = 0;
            for (int i = sub; i < len; i += 8 * kSumWaves) {
                int64_t y[8], s2 = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    y[k] = static_cast<int64_t>(r[i + k * kSumWaves < len ? i + k * kSumWaves : i]);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if (i + k * kSumWaves >= len) y[k] = 0;
                    s1 += y[k];
                    s2 += y[k] * (i + k * kSumWaves);
                }
                a2 += s2;
            }
            a1 = s1;
        }
        for (int o = 1; o < kSumWaves; o <<= 1) {
            a1 += shfl_xor_i128(a1, o);
            a2 += shfl_xor_i128(a2, o);
        }
        if (sub == 0) {
            s_sum[0][blk] = a1;
            s_sum[1][blk] = a2;
        }
    }
    __syncthreads();
    if (w == kBlkThreads / 64 - 1) {  // scan over the 64 blocks
        const i128 a1 = s_sum[0][lane];
        const i128 a2 = s_sum[1][lane] + a1 * static_cast<i128>(q0 + static_cast<int64_t>(lane) * B);  // q = first + i
        i128 s1 = a1, s2 = a2;  // inclusive
        for (int o = 1; o < 64; o <<= 1) {
            const i128 x1 = shfl_up_i128(s1, o), x2 = shfl_up_i128(s2, o);
            if (lane >= o) {
                s1 += x1;
                s2 += x2;
            }
        }
        if (b0 + lane <= JB) {
            p1[b0 + lane] = s1 - a1;
            p2[b0 + lane] = s2 - a2;
        }
        if (lane == 63) {
            c1[blockIdx.x] = s1;
            c2[blockIdx.x] = s2;
        }
    }
    // vertices: lane = block, the waves take one in turn; the upper hull's, then
    // the lower one's without the two ends they share
    const int64_t b = b0 + lane;
    if (b >= JB) return;
    const int nu = s_n[0][lane], nl = s_n[1][lane];
    const int total = nu + (nl > 2 ? nl - 2 : 0);
    if (nu > kHullCand || nl > kHullCand || total > h.slots || s_big[lane]) {
        if (w == 0) h.nv[b] = kHullScan;
        return;
    }
    if (w == 0) h.nv[b] = static_cast<uint8_t>(total);
    for (int k = w; k < total; k += kBlkThreads / 64) {
        const int i = k < nu ? s_list[0][k * 64 + lane] : s_list[1][(k - nu + 1) * 64 + lane];
        h.y[hull_at(h.slots, b, k)] = row[i];
        h.x[hull_at(h.slots, b, k)] = static_cast<uint8_t>(i);
    }
}

// Sums without hulls, for block sizes above kHullMaxB: a workgroup per block,
// then the exclusive scan inside each chunk.
template <class T>
__global__ __launch_bounds__(kSmThreads) void k_sm_sums(const T* __restrict__ v, int64_t n, int32_t B,
                                                        i128* __restrict__ p1, i128* __restrict__ p2) {
    __shared__ i128 s1[kSmThreads / 64], s2[kSmThreads / 64];
    const int tid = threadIdx.x;
    const int64_t q0 = static_cast<int64_t>(blockIdx.x) * B;
    const int64_t q1 = (q0 + B < n) ? q0 + B : n;
    i128 a1 = 0, a2 = 0;
    for (int64_t q = q0 + tid; q < q1; q += kSmThreads) {
        const i128 y = wide<T>(v[q]);
        a1 += y;
        a2 += y * static_cast<i128>(q);
    }
    a1 = wave_sum(a1);
    a2 = wave_sum(a2);
    if ((tid & 63) == 0) {
        s1[tid >> 6] = a1;
        s2[tid >> 6] = a2;
    }
    __syncthreads();
    if (tid == 0) {
        for (int k = 1; k < kSmThreads / 64; ++k) {
            a1 += s1[k];
            a2 += s2[k];
        }
        p1[blockIdx.x] = a1;
        p2[blockIdx.x] = a2;
    }
}
__global__ __launch_bounds__(kPfxChunk) void k_sm_chunk_pfx(int64_t JB, i128* __restrict__ p1, i128* __restrict__ p2,
                                                             i128* __restrict__ c1, i128* __restrict__ c2) {
    __shared__ i128 s1[kPfxChunk], s2[kPfxChunk];
    const int tid = threadIdx.x;
    const int64_t p = static_cast<int64_t>(blockIdx.x) * kPfxChunk + tid;
    const i128 a1 = p < JB ? p1[p] : static_cast<i128>(0), a2 = p < JB ? p2[p] : static_cast<i128>(0);
    s1[tid] = a1;
    s2[tid] = a2;
    __syncthreads();
    for (int o = 1; o < kPfxChunk; o <<= 1) {  // inclusive scan
        const i128 x1 = (tid >= o) ? s1[tid - o] : static_cast<i128>(0);
        const i128 x2 = (tid >= o) ? s2[tid - o] : static_cast<i128>(0);
        __syncthreads();
        s1[tid] += x1;
        s2[tid] += x2;
        __syncthreads();
    }
    if (p <= JB) {
        p1[p] = s1[tid] - a1;
        p2[p] = s2[tid] - a2;
    }
    if (tid == kPfxChunk - 1) {
        c1[blockIdx.x] = s1[tid];
        c2[blockIdx.x] = s2[tid];
    }
}
// exclusive scan of C chunk totals in place (one workgroup, serial chunks)
constexpr int kChunkScanThreads = 1024;
__global__ __launch_bounds__(kChunkScanThreads) void k_sm_chunk_scan(i128* __restrict__ c1, i128* __restrict__ c2,
                                                              int64_t C) {
    __shared__ i128 s1[kChunkScanThreads], s2[kChunkScanThreads];
    const int tid = threadIdx.x;
    const int64_t per = (C + kChunkScanThreads - 1) / kChunkScanThreads;
    const int64_t b0 = tid * per;
    const int64_t b1 = (b0 + per < C) ? b0 + per : C;
    i128 a1 = 0, a2 = 0;
    for (int64_t i = b0; i < b1; ++i) {
        a1 += c1[i];
        a2 += c2[i];
    }
    s1[tid] = a1;
    s2[tid] = a2;
    __syncthreads();
    for (int o = 1; o < kChunkScanThreads; o <<= 1) {
        const i128 x1 = (tid >= o) ? s1[tid - o] : static_cast<i128>(0);
        const i128 x2 = (tid >= o) ? s2[tid - o] : static_cast<i128>(0);
        __syncthreads();
        s1[tid] += x1;
        s2[tid] += x2;
        __syncthreads();
    }
    i128 r1 = s1[tid] - a1, r2 = s2[tid] - a2;  // exclusive
    for (int64_t i = b0; i < b1; ++i) {
        const i128 t1 = c1[i], t2 = c2[i];
        c1[i] = r1;
        c2[i] = r2;
        r1 += t1;
        r2 += t2;
    }
}

// The same evaluation from prefix sums and hulls, S consecutive starts per
// workgroup (m = U * B, S = 8 / U): their candidates lie in a window of
// (S - 1 + 29) U blocks, whose vertices are staged in LDS.  Each thread takes
// (start, candidate, block) triples and raises the candidate's D.  A candidate
// that D does not settle gets its H from a wave, and one that this does not
// settle is read value by value.
constexpr int kSplitMaxU = 8;
constexpr int kCandUnitSum = 162;
inline __host__ __device__ int split_starts(int U) { return U >= kSplitMaxU ? 1 : 8 / U; }
inline __host__ __device__ int split_window(int U) { return (split_starts(U) - 1 + 29) * U; }
inline size_t split_lds(int U, int32_t slots) { return static_cast<size_t>(split_window(U)) * (slots * 9 + 1); }

template <class T>
__global__ __launch_bounds__(kSmThreads) void k_sm_split_hull(const T* __restrict__ v, int64_t n, int32_t m, int64_t J,
                                                              int U, SmPrefix pf, SmHull h,
                                                              int32_t* __restrict__ best_end,
                                                              double* __restrict__ best_cost) {
    constexpr int kS = 8, kTasks = kS * kMaxCand;
    extern __shared__ double s_y[];  // [slots][W], then x [slots][W], nv [W]
    __shared__ double s_t[kTasks][2];
    __shared__ unsigned long long s_D[kTasks];  // bits of non-negative doubles: ordered as integers
    __shared__ int32_t s_bits[kTasks], s_scan[kTasks], s_fast[kTasks];
    __shared__ int s_list[2][kTasks], s_cnt[2];
    __shared__ uint16_t s_unit[kCandUnitSum];  // of one start's candidates' units: candidate, unit of it << 4
    __shared__ int64_t s_mx[kSmThreads / 64];
    __shared__ FitLds L;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int S = split_starts(U), W = split_window(U);
    uint8_t* s_x = reinterpret_cast<uint8_t*>(s_y + h.slots * W);
    uint8_t* s_nv = s_x + h.slots * W;
    const int64_t j0 = static_cast<int64_t>(blockIdx.x) * S;
    const int64_t bw = j0 * U;  // first block of the window
    int most = 0;
    for (int i = tid; i < W; i += kSmThreads) {
        const int c = bw + i < pf.JB ? h.nv[bw + i] : 0;
        s_nv[i] = static_cast<uint8_t>(c);
        most = c != kHullScan && c > most ? c : most;
    }
    if (tid < 2) s_cnt[tid] = 0;
    if (tid < kCandUnitSum) {
        int k = 0;
#pragma unroll
        for (int c = 1; c < kMaxCand; ++c) k += tid >= kCandCum[c];
        s_unit[tid] = static_cast<uint16_t>(k | (tid - kCandCum[k]) << 4);
    }
    // task q * 14 + k: candidate k of start j0 + q
    const int tq = tid / kMaxCand, tk = tid % kMaxCand;
    const int64_t cur = (j0 + tq) * m, size = static_cast<int64_t>(kCandUnits[tk]) * m;
    const bool live = tid < S * kMaxCand && cur + size <= n;
    if (tid < kTasks) {
        s_D[tid] = 0;
        s_bits[tid] = live ? 0 : -1;
        s_scan[tid] = 0;
        if (live) {
            bool fast;
            range_line<T>(pf, cur, cur + size, s_t[tid][0], s_t[tid][1], fast);
            s_fast[tid] = fast;
            s_scan[tid] = !fast;
        }
    }
    const int rows = __syncthreads_or(most > 16) ? h.slots : h.slots < 16 ? h.slots : 16;
    const uint32_t rcp_w = 0xFFFFFFFFu / static_cast<uint32_t>(W) + 1u;  // exact for i * W < 2^32
    for (int i = tid; i < rows * W; i += kSmThreads) {
        const int k = static_cast<int>(__umulhi(static_cast<uint32_t>(i), rcp_w)), b = i - k * W;
        if (bw + b < pf.JB) {  // slots past a block's vertices hold whatever was there and are not read below
            s_y[i] = h.y[hull_at(h.slots, bw + b, k)];
            s_x[i] = h.x[hull_at(h.slots, bw + b, k)];
        }
    }
    __syncthreads();
    const int per = kCandUnitSum * U;  // blocks of one start's candidates
    const uint32_t rcp = 0xFFFFFFFFu / static_cast<uint32_t>(per) + 1u;
    for (int t = tid; t < S * per; t += kSmThreads) {
        const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(t), rcp)), r = t - q * per;
        const int x = s_unit[U == 1 ? r : r / U];
        const int u = (x >> 4) * U + (U == 1 ? 0 : r % U), b = q * U + u;
        const int task = q * kMaxCand + (x & 15);
        if (s_bits[task] < 0 || s_scan[task]) continue;
        const int nv = s_nv[b];
        if (nv == kHullScan) {
            s_scan[task] = 1;
            continue;
        }
        const double D = hull_far(s_y + b, s_x + b, W, nv, u * pf.B, s_t[task][0], s_t[task][1]);
        atomicMax(&s_D[task], static_cast<unsigned long long>(__double_as_longlong(D)));
    }
    __syncthreads();
    if (live) {
        const int32_t b = s_scan[tid] ? -1
                                      : hull_bits(__longlong_as_double(static_cast<long long>(s_D[tid])), 0.0,
                                                  s_t[tid][0], s_t[tid][1], size);
        if (b < 0) s_list[s_scan[tid]][atomicAdd(&s_cnt[s_scan[tid]], 1)] = tid;
        else s_bits[tid] = b;
    }
    __syncthreads();
    const int open = s_cnt[0];
    for (int i = w; i < open; i += kSmThreads / 64) {  // a wave each: H
        const int task = s_list[0][i], k = task % kMaxCand, q = task / kMaxCand;
        const double t0 = s_t[task][0], t1 = s_t[task][1];
        double H = 0.0;
        for (int u = lane; u < kCandUnits[k] * U; u += 64) {
            const int b = q * U + u;
            H = __builtin_fmax(H, hull_low(s_y + b, s_x + b, W, s_nv[b], u * pf.B, t0, t1));
        }
        for (int o = 32; o > 0; o >>= 1) H = __builtin_fmax(H, __shfl_xor(H, o, 64));
        const int32_t b = hull_bits(__longlong_as_double(static_cast<long long>(s_D[task])), H, t0, t1,
                                    static_cast<int64_t>(kCandUnits[k]) * m);
        if (lane == 0) {
            if (b < 0) s_list[1][atomicAdd(&s_cnt[1], 1)] = task;
            else s_bits[task] = b;
        }
    }
    __syncthreads();
    for (int i = 0; i < s_cnt[1]; ++i) {  // read by the whole workgroup
        const int task = s_list[1][i];
        const int64_t c = (j0 + task / kMaxCand) * m, z = static_cast<int64_t>(kCandUnits[task % kMaxCand]) * m;
        const int64_t mx = wave_max(
            scan_err<T>(v + c, tid, z, kSmThreads, s_t[task][0], s_t[task][1], s_fast[task] != 0));
        if (lane == 0) s_mx[w] = mx;
        __syncthreads();
        if (tid == 0) {
            int64_t r = s_mx[0];
            for (int x = 1; x < kSmThreads / 64; ++x) r = s_mx[x] > r ? s_mx[x] : r;
            s_bits[task] = bits_of(r);
        }
        __syncthreads();
    }
    if (live) {
        const double c = cost_of(size, s_bits[tid]);
        s_t[tid][0] = c / static_cast<double>(size);
        s_t[tid][1] = c;
    }
    __syncthreads();
    if (tid < S && j0 + tid < J && s_bits[tid * kMaxCand] >= 0) {  // smallest cost per value, the first on ties
        int at = 0;
        for (int k = 1; k < kMaxCand && s_bits[tid * kMaxCand + k] >= 0; ++k)
            if (s_t[tid * kMaxCand + k][0] < s_t[tid * kMaxCand + at][0]) at = k;
        best_end[j0 + tid] = static_cast<int32_t>((j0 + tid) * m + static_cast<int64_t>(kCandUnits[at]) * m);
        best_cost[j0 + tid] = s_t[tid * kMaxCand + at][1];
    }
    // the column's last start may have fewer than m values: one partition [cur, n)
    const int64_t last = (J - 1) * m;
    if (J - 1 >= j0 && J - 1 < j0 + S && n - last < m) {
        const double c = wg_cost<T>(v, last, n, L);
        if (tid == 0) {
            best_end[J - 1] = static_cast<int32_t>(n);
            best_cost[J - 1] = c;
        }
    }
}

// ---- chain: mark the entries that a walk from entry 0 reaches ----------------
// next[i] > i is the entry after i (J or more: the end).  k_sm_chain_exit: a
// workgroup per chunk of kChain entries replaces next by the first entry past
// the chunk, by pointer doubling in LDS; k_sm_chain_walk hops from chunk to
// chunk (one dependent load each) and notes where the walk enters each;
// k_sm_chain_mark marks a chunk's entries from there, again by doubling.  Three
// launches where doubling over the whole list took 2 log2(J).
constexpr int kChainThreads = 1024;
constexpr int kChainPer = 8;
constexpr int kChain = kChainThreads * kChainPer;

// one doubling step over the chunk's LDS copy; true while some entry is inside
__device__ __forceinline__ bool chain_double(int32_t* s_j, int32_t cnt) {
    int32_t t[kChainPer];
    bool inside = false;
#pragma unroll
    for (int q = 0; q < kChainPer; ++q) {
        const int32_t i = threadIdx.x + q * kChainThreads;
        t[q] = i < cnt ? s_j[i] : cnt;
        if (t[q] < cnt) t[q] = s_j[t[q]];
        inside = inside || t[q] < cnt;
    }
    const bool any = __syncthreads_or(inside);
#pragma unroll
    for (int q = 0; q < kChainPer; ++q) {
        const int32_t i = threadIdx.x + q * kChainThreads;
        if (i < cnt) s_j[i] = t[q];
    }
    __syncthreads();
    return any;
}

// next[] of entry i: its target entry, J past the end
struct ChainSplit {  // split: best_end[i] / m where that is an entry
    const int32_t* best_end;
    int64_t J;
    int32_t m;
    __device__ int64_t operator()(int64_t i) const {
        const uint32_t e = static_cast<uint32_t>(best_end[i]), j = e / static_cast<uint32_t>(m);
        return (j * static_cast<uint32_t>(m) == e && j < J) ? j : J;
    }
};
struct ChainMerge {  // merge: the group that starts at partition i ends before partition gend[i]
    const int32_t* gend;
    __device__ int64_t operator()(int64_t i) const { return gend[i]; }
};

template <class F>
__global__ __launch_bounds__(kChainThreads) void k_sm_chain_exit(F next, int64_t J, int32_t* __restrict__ out) {
    __shared__ int32_t s_j[kChain];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kChain;
    const int32_t cnt = static_cast<int32_t>(J - base < kChain ? J - base : kChain);
    // targets relative to the chunk; one past it is kept as it is (>= cnt) and
    // never followed inside
    bool inside = false;
    for (int32_t i = threadIdx.x; i < cnt; i += kChainThreads) {
        s_j[i] = static_cast<int32_t>(next(base + i) - base);
        inside = inside || s_j[i] < cnt;
    }
    bool any = __syncthreads_or(inside);
    while (any) any = chain_double(s_j, cnt);
    for (int32_t i = threadIdx.x; i < cnt; i += kChainThreads) out[base + i] = static_cast<int32_t>(base + s_j[i]);
}
__global__ void k_sm_chain_walk(const int32_t* __restrict__ exits, int64_t J, int64_t chunks,
                                int32_t* __restrict__ entry) {
    for (int64_t c = threadIdx.x; c < chunks; c += blockDim.x) entry[c] = -1;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t e = 0;
        while (e < J) {
            entry[e / kChain] = static_cast<int32_t>(e);
            e = exits[e];
        }
    }
}
template <class F>
__global__ __launch_bounds__(kChainThreads) void k_sm_chain_mark(F next, int64_t J, const int32_t* __restrict__ entry,
                                                                 int32_t* __restrict__ mark) {
    __shared__ int32_t s_j[kChain];
    __shared__ uint8_t s_m[kChain];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kChain;
    const int32_t cnt = static_cast<int32_t>(J - base < kChain ? J - base : kChain);
    const int32_t e = entry[blockIdx.x];
    bool inside = false;
    for (int32_t i = threadIdx.x; i < cnt; i += kChainThreads) {
        s_j[i] = static_cast<int32_t>(next(base + i) - base);
        s_m[i] = e >= 0 && base + i == e;
        inside = inside || s_j[i] < cnt;
    }
    bool any = __syncthreads_or(inside) && e >= 0;
    while (any) {  // entries on the walk mark their targets, then every target doubles
        for (int32_t i = threadIdx.x; i < cnt; i += kChainThreads)
            if (s_m[i] && s_j[i] < cnt) s_m[s_j[i]] = 1;
        __syncthreads();
        any = chain_double(s_j, cnt);
    }
    for (int32_t i = threadIdx.x; i < cnt; i += kChainThreads) mark[base + i] = s_m[i];
}

// exclusive scan of mark[] into pos[]; *count = total (one workgroup)
constexpr int kScan = 1024;
__global__ __launch_bounds__(kScan) void k_sm_scan(const int32_t* __restrict__ mark, int64_t J,
                                                   int32_t* __restrict__ pos, int64_t* __restrict__ count) {
    __shared__ int64_t s[kScan];
    const int tid = threadIdx.x;
    const int64_t chunk = (J + kScan - 1) / kScan;
    const int64_t b0 = tid * chunk;
    const int64_t b1 = (b0 + chunk < J) ? b0 + chunk : J;
    int64_t local = 0;
    for (int64_t i = b0; i < b1; ++i) local += mark[i];
    s[tid] = local;
    __syncthreads();
    for (int o = 1; o < kScan; o <<= 1) {
        const int64_t y = (tid >= o) ? s[tid - o] : 0;
        __syncthreads();
        s[tid] += y;
        __syncthreads();
    }
    int64_t acc = s[tid] - local;
    for (int64_t i = b0; i < b1; ++i) {
        pos[i] = static_cast<int32_t>(acc);
        acc += mark[i];
    }
    if (tid == kScan - 1) *count = s[tid];
}
// Exclusive scan of a long flag array: k_sm_scan_local scans kScanTile
// entries per workgroup (16 consecutive per thread) and writes the tile
// totals; k_sm_scan (one workgroup) scans the totals into tile offsets and the
// grand total; k_sm_scan_add adds the offsets.
constexpr int kScanPer = 16;
constexpr int kScanTile = kSmThreads * kScanPer;
__global__ __launch_bounds__(kSmThreads) void k_sm_scan_local(const int32_t* __restrict__ mark, int64_t N,
                                                              int32_t* __restrict__ pos,
                                                              int32_t* __restrict__ tile_tot) {
    __shared__ int32_t s[kSmThreads];
    const int tid = threadIdx.x;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + static_cast<int64_t>(tid) * kScanPer;
    int32_t f[kScanPer];
    int32_t sum = 0;
#pragma unroll
    for (int q = 0; q < kScanPer; ++q) {
        f[q] = (base + q < N) ? mark[base + q] : 0;
        sum += f[q];
    }
    s[tid] = sum;
    __syncthreads();
    for (int o = 1; o < kSmThreads; o <<= 1) {
        const int32_t y = (tid >= o) ? s[tid - o] : 0;
        __syncthreads();
        s[tid] += y;
        __syncthreads();
    }
    int32_t acc = s[tid] - sum;
#pragma unroll
    for (int q = 0; q < kScanPer; ++q) {
        if (base + q < N) pos[base + q] = acc;
        acc += f[q];
    }
    if (tid == kSmThreads - 1) tile_tot[blockIdx.x] = s[tid];
}
__global__ void k_sm_scan_add(int32_t* __restrict__ pos, int64_t N, const int32_t* __restrict__ tile_off) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < N) pos[i] += tile_off[i / kScanTile];
}

// Marked entry i becomes entry p of the next list; entry 0's length is
// reported to pinned memory (host[1]).
struct EmitSplit {
    const int32_t* best_end;
    const double* best_cost;
    int32_t m;
    int32_t *st, *en;
    double* cost;
    int64_t* host;
    __device__ void operator()(int64_t i, int64_t p) const {
        const int32_t s = static_cast<int32_t>(i * m), e = best_end[i];
        st[p] = s;
        en[p] = e;
        cost[p] = best_cost[i];
        if (p == 0) host[1] = e - s;
    }
};
struct EmitGroups {
    const int32_t* gend;
    const double* gcost;
    const int32_t *st, *en;
    int32_t *ost, *oen;
    double* ocost;
    int64_t* host;
    __device__ void operator()(int64_t i, int64_t p) const {
        const int32_t s = st[i], e = en[gend[i] - 1];
        ost[p] = s;
        oen[p] = e;
        ocost[p] = gcost[i];
        if (p == 0) host[1] = e - s;
    }
};
template <class E>
__global__ void k_sm_emit(const int32_t* __restrict__ mark, const int32_t* __restrict__ pos, int64_t N, E emit) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < N && mark[i]) emit(i, pos[i]);
}

// Chain, scan and emission of a list of at most kChain entries by one
// workgroup: one launch instead of seven (4-5 us each with its gap), which were
// half of a 2^16-value call.
template <class F, class E>
__global__ __launch_bounds__(kChainThreads) void k_sm_chain_small(F next, E emit, int32_t N, int64_t* __restrict__ host) {
    __shared__ int32_t s_j[kChain];
    __shared__ uint8_t s_m[kChain];
    __shared__ int32_t s_w[kChainThreads / 64 + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    bool inside = false;
    for (int32_t i = tid; i < N; i += kChainThreads) {
        s_j[i] = static_cast<int32_t>(next(i));
        s_m[i] = i == 0;
        inside = inside || s_j[i] < N;
    }
    bool any = __syncthreads_or(inside);
    while (any) {
        for (int32_t i = tid; i < N; i += kChainThreads)
            if (s_m[i] && s_j[i] < N) s_m[s_j[i]] = 1;
        __syncthreads();
        any = chain_double(s_j, N);
    }
    // positions: thread tid counts entries tid * kChainPer ...
    int32_t sum = 0;
#pragma unroll
    for (int q = 0; q < kChainPer; ++q) {
        const int32_t i = tid * kChainPer + q;
        sum += i < N ? s_m[i] : 0;
    }
    int32_t incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    if (lane == 63) s_w[w] = incl;
    __syncthreads();
    if (tid == 0) {
        int32_t acc = 0;
        for (int k = 0; k < kChainThreads / 64; ++k) {
            const int32_t t = s_w[k];
            s_w[k] = acc;
            acc += t;
        }
        host[0] = acc;
    }
    __syncthreads();
    int32_t at = s_w[w] + incl - sum;
#pragma unroll
    for (int q = 0; q < kChainPer; ++q) {
        const int32_t i = tid * kChainPer + q;
        if (i < N && s_m[i]) emit(i, at++);
    }
}

// ---- merge -------------------------------------------------------------------
// The group that starts at partition e (CpuPartitioner.cuh:207-236): it takes
// in partition j while the refitted whole costs less than the group so far and
// j apart.  Whether the walk starts a group at e or not, what the group would
// be depends on e alone, so all are grown at once, a wave each; gend[e] is the
// first partition after the group, gcost[e] its cost.  The lines of the next
// kGrowLook candidates are computed by as many lanes at once; one candidate's
// residuals take the hulls of its blocks, a block per lane.
//
// Total work.  Every candidate of every start takes its whole range again: P starts
// x candidates of a group x blocks of a group / 64 steps.  A group mostly ends by
// 46341 values, where the cost model's int32 n * (n - 1) wraps: 12 candidates of 362
// blocks at m = 128, but 1600 at m = 1 (a split partition has up to 29 m values); and
// values that are all near 0 fit any line, so their group takes in the whole
// column.  Hence kGrowSteps, after which a wave stops; of the groups left open only
// those that the walk reaches count, and they are grown on by the whole GPU.  The
// bound: P x kGrowSteps steps here, then the walk's own candidates x blocks / 64 steps
// over up to kMoreCand waves.  A candidate counts as a step for every 64 blocks and one for
// every 256 values (it may come to be read): m = 32 and above end here (4900 at 32),
// which are 3 times as fast so (2^21 noisy values, bound 4096 against 8192: m = 32
// 11.6 and 4.1 ms, m = 1 152 and 236 ms).
constexpr int kGrowLook = 16;
constexpr float kGrowSteps = 6144.0f;

// Bit width of the residuals of line t0, t1 over [gs, ge), computed by a
// wave (gs a block start, ge one or n).
template <class T>
__device__ __forceinline__ int32_t range_bits(const T* __restrict__ v, int64_t gs, int64_t ge, double t0, double t1,
                                              bool fast, const SmPrefix& pf, const SmHull& h, int lane) {
    const int64_t len = ge - gs;
    int32_t bits = -1;
    if (fast && h.slots > 0) {
        const int64_t ib = block_of(pf, gs), ie = (ge == pf.n) ? pf.JB : block_of(pf, ge);
        double D = 0.0;
        int64_t mx = 0;  // of blocks read value by value
        bool settled = true, read = false;
        for (int64_t b0 = ib; b0 < ie; b0 += 64) {
            const int64_t b = b0 + lane;
            int nv = b < ie ? h.nv[b] : 0;
            uint64_t odd = __ballot(nv == kHullScan);
            if (__popcll(odd) > 8) {  // mostly such blocks: one pass over the range is faster
                settled = false;
                break;
            }
            if (nv == kHullScan) nv = 0;
            const int64_t at = hull_at(h.slots, b < ie ? b : ib, 0);
            D = __builtin_fmax(D, hull_far(h.y + at, h.x + at, 64, nv, static_cast<int32_t>(b - ib) * pf.B, t0, t1));
            while (odd) {  // wave-uniform
                read = true;
                const int64_t q = (b0 + __builtin_ctzll(odd)) * pf.B;
                odd &= odd - 1;
                const int64_t hi = q + pf.B < ge ? q + pf.B : ge;
                const int64_t a = scan_err<T>(v + gs, q - gs + lane, hi - gs, 64, t0, t1, true);
                mx = a > mx ? a : mx;
            }
        }
        for (int o = 32; o > 0; o >>= 1) D = __builtin_fmax(D, __shfl_xor(D, o, 64));
        bits = settled ? hull_bits(D, 0.0, t0, t1, len) : -1;
        if (settled && bits < 0) {
            double H = 0.0;
            for (int64_t b = ib + lane; b < ie; b += 64) {
                const int64_t at = hull_at(h.slots, b, 0);
                const int nv = h.nv[b];
                H = __builtin_fmax(H, hull_low(h.y + at, h.x + at, 64, nv == kHullScan ? 0 : nv,
                                               static_cast<int32_t>(b - ib) * pf.B, t0, t1));
            }
            for (int o = 32; o > 0; o >>= 1) H = __builtin_fmax(H, __shfl_xor(H, o, 64));
            bits = hull_bits(D, H, t0, t1, len);
        }
        if (bits >= 0 && read) {
            mx = wave_max(mx);
            bits = bits_of(mx) > bits ? bits_of(mx) : bits;
        }
    }
    return bits >= 0 ? bits : bits_of(wave_max(scan_err<T>(v + gs, lane, len, 64, t0, t1, fast)));
}

// *more (pinned): set where a group is left open after kGrowSteps steps; its
// gcost is then negative, and gend the first partition not yet asked.
template <class T>
__global__ __launch_bounds__(kSmThreads) void k_sm_grow(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                        const int32_t* __restrict__ en,
                                                        const double* __restrict__ cost, int64_t P, SmPrefix pf,
                                                        SmHull h, int32_t* __restrict__ gend,
                                                        double* __restrict__ gcost, int64_t* __restrict__ more) {
    const int lane = threadIdx.x & 63;
    const int64_t e = static_cast<int64_t>(blockIdx.x) * (kSmThreads / 64) +
                      __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (e >= P) return;
    const int64_t gs = st[e];
    double gc = cost[e];
    int64_t j = e + 1;
    bool open = true;
    const float per = 1.0f / 256.0f + 1.0f / (64.0f * static_cast<float>(pf.B));
    float steps = 0.0f;
    while (open && j < P && steps < kGrowSteps) {
        double lt0 = 0.0, lt1 = 0.0, lc = 0.0;
        int32_t le = 0;
        bool lf = false;
        if (lane < kGrowLook && j + lane < P) {
            le = en[j + lane];
            lc = cost[j + lane];
            range_line<T>(pf, gs, le, lt0, lt1, lf);
        }
        const int look = P - j < kGrowLook ? static_cast<int>(P - j) : kGrowLook;
        for (int c = 0; c < look && open && steps < kGrowSteps; ++c) {
            const int64_t ge = __shfl(le, c, 64);
            const double merged =
                cost_of(ge - gs, range_bits<T>(v, gs, ge, __shfl(lt0, c, 64), __shfl(lt1, c, 64),
                                               __shfl(static_cast<int>(lf), c, 64) != 0, pf, h, lane));
            steps += per * static_cast<float>(static_cast<int32_t>(ge - gs));
            open = merged < gc + __shfl(lc, c, 64);
            if (open) {
                gc = merged;
                ++j;
            }
        }
    }
    if (lane == 0) {
        const bool left = open && j < P;
        gend[e] = static_cast<int32_t>(j);
        gcost[e] = left ? -gc : gc;  // a cost is at least 80
        if (left) *more = 1;
    }
}

// The open group that the walk is at (e = P: none left).
struct SmOpen {
    int64_t e, j;  // its start, the first partition not yet asked
    double gc;
};

// How many candidates the open group is asked for next: as many as it holds, so
// that what is asked past its end stays in proportion (2^20 noisy values, m = 8: 81 ms
// with all of kMoreCand at once, 25 so).
constexpr int kMoreCand = 4096;
__device__ __forceinline__ int more_cand(const SmOpen& o, int64_t P) {
    int64_t n = o.j - o.e;
    n = n < 64 ? 64 : n > kMoreCand ? kMoreCand : n;
    return static_cast<int>(n < P - o.j ? n : P - o.j);
}

// Costs of the open group with each of the next candidates taken in, a wave
// each, as if all before were.
template <class T>
__global__ __launch_bounds__(kSmThreads) void k_sm_more(const T* __restrict__ v, const int32_t* __restrict__ st,
                                                        const int32_t* __restrict__ en, int64_t P, SmPrefix pf,
                                                        SmHull h, const SmOpen* __restrict__ open,
                                                        double* __restrict__ merged) {
    const int q = static_cast<int>(blockIdx.x) * (kSmThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const SmOpen o = *open;
    if (o.e >= P || q >= more_cand(o, P)) return;
    const int64_t gs = st[o.e], ge = en[o.j + q];
    double t0, t1;
    bool fast;
    range_line<T>(pf, gs, ge, t0, t1, fast);
    const double c = cost_of(ge - gs, range_bits<T>(v, gs, ge, t0, t1, fast, pf, h, threadIdx.x & 63));
    if ((threadIdx.x & 63) == 0) merged[q] = c;
}

// Takes in the candidates of k_sm_more up to the first that does not pay; where
// the group ends there, the walk goes on to the next open one.  first: the walk is
// at partition 0.  *more (pinned): 0 when it has reached the end.  One workgroup.
constexpr int kWalkThreads = 1024;
constexpr int kWalkWin = 4096;
__global__ __launch_bounds__(kWalkThreads) void k_sm_walk(const double* __restrict__ cost,
                                                          const double* __restrict__ merged, int64_t P, bool first,
                                                          int32_t* __restrict__ gend, double* __restrict__ gcost,
                                                          SmOpen* __restrict__ open, int64_t* __restrict__ more) {
    __shared__ int32_t s_next[kWalkWin];  // gend, negative where open; of the entries from wb on
    __shared__ int s_end;
    const int tid = threadIdx.x;
    int64_t e = 0;  // the same in every thread, as all below
    if (!first) {
        const SmOpen o = *open;
        e = o.e;
        if (e >= P) return;
        const int n = more_cand(o, P);
        if (tid == 0) s_end = n;
        __syncthreads();
        for (int c = tid; c < n; c += kWalkThreads)
            if (!(merged[c] < (c == 0 ? o.gc : merged[c - 1]) + cost[o.j + c])) atomicMin(&s_end, c);
        __syncthreads();
        const int end = s_end;
        const double gc = end == 0 ? o.gc : merged[end - 1];
        if (end == n && o.j + n < P) {  // still open
            if (tid == 0) {
                open->j = o.j + n;
                open->gc = gc;
            }
            return;
        }
        if (tid == 0) {
            gend[e] = static_cast<int32_t>(o.j + end);
            gcost[e] = gc;
        }
        e = o.j + end;
    }
    for (int64_t wb = e - kWalkWin; e < P;) {
        if (e >= wb + kWalkWin) {
            __syncthreads();
            wb = e;
            for (int q = tid; q < kWalkWin && wb + q < P; q += kWalkThreads)
                s_next[q] = gcost[wb + q] < 0.0 ? -gend[wb + q] : gend[wb + q];
            __syncthreads();
        }
        const int32_t next = s_next[e - wb];
        if (next < 0) {
            if (tid == 0) *open = SmOpen{e, -next, -gcost[e]};
            return;
        }
        e = next;
    }
    if (tid == 0) {
        open->e = P;
        *more = 0;
    }
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

unsigned blocks(int64_t n, int b) { return static_cast<unsigned>((n + b - 1) / b); }

// Scratch of one split/merge call, kept per device between calls and grown
// when a larger column needs more (a per-call hipMalloc/hipFree pair costs
// hundreds of microseconds and the free synchronises the device).  Held
// until the process ends; one above kSmKeep bytes (a column of about 2^28 values
// at minimum size 128) is given back by split_merge_release.  The lock covers a call
// and the launch of its caller's copy of the boundaries.
constexpr int64_t kSmKeep = int64_t(1) << 30;
SharedScratch& sm_scratch(int device) {
    static std::mutex table_mu;
    static std::map<int, SharedScratch*>* table = new std::map<int, SharedScratch*>();  // never freed: used until exit
    std::lock_guard<std::mutex> g(table_mu);
    SharedScratch*& e = (*table)[device];
    if (!e) e = new SharedScratch();
    return *e;
}

}  // namespace

// Partition d_values[0, n), n > 0, on the device; the boundaries stay in the
// scratch, whose lock goes to the caller.
int gpu_split_merge(int dtype, const void* d_values, int64_t n, int32_t m, SplitMergeResult* out, hipStream_t s) {
    if (m <= 0 || m > (1 << 20)) return fail(GLC_ERR_INVALID_ARG, "split/merge minimum size must be in [1, 2^20]");
    const int64_t J = (n + m - 1) / m;
    // blocks: B = m up to kHullMaxB; above, the largest divisor of m from 32
    // to kHullMaxB with m / B <= kSplitMaxU (wide enough to make hulls pay, few
    // enough for the split window).  No such divisor: B = m, sums only.
    int32_t B = m;
    if (m > kHullMaxB)
        for (int32_t d = kHullMaxB; d >= 32; --d)
            if (m % d == 0 && m / d <= kSplitMaxU) {
                B = d;
                break;
            }
    const bool hulls = B <= kHullMaxB;
    const int32_t slots = hulls ? std::min<int32_t>(kHullSlots, B) : 0;
    const int U = m / B;
    const int64_t JB = (n + B - 1) / B;
    // scratch: best_end, exits, mark, pos, st x2, en x2, gend (int32 x J each);
    // best_cost, cost x2, gcost (double x J each); the open group (256 bytes); block
    // prefixes p1, p2 (i128 x (JB + 1)) and chunk offsets c1, c2 (i128 x C); scan
    // tile totals and offsets (int32 x T), chain entries (int32); hull vertices
    // y (double), x (byte) x slots and counts (byte) per block, 64 blocks at a time
    const int64_t i4 = align_up(J * 4, 256), d8 = align_up(J * 8, 256);
    const int64_t C = (JB + 1 + kPfxChunk - 1) / kPfxChunk;
    const int64_t q16 = align_up((JB + 1) * 16, 256), c16 = align_up(C * 16, 256);
    const int64_t T = (J + kScanTile - 1) / kScanTile;
    const int64_t t4 = align_up(T * 4, 256);
    const int64_t jb64 = align_up(JB, 64);
    const int64_t hy = align_up(jb64 * slots * 8, 256), hx = align_up(jb64 * slots, 256), hn = align_up(jb64, 256);
    const int64_t bytes = 9 * i4 + 4 * d8 + 256 + 2 * q16 + 2 * c16 + 3 * t4 + (hulls ? hy + hx + hn : 0);
    int dev = 0;
    GLC_HIP(hipGetDevice(&dev));
    HostWords host;
    if (!host.p) return fail(GLC_ERR_OOM, "pinned host allocation failed");
    SharedScratch& sc = sm_scratch(dev);
    std::unique_lock<std::mutex> scratch_lock(sc.mu);
    const int ac = scratch_acquire(sc, bytes, s);
    if (ac) return ac;
    char* p = static_cast<char*>(sc.p);
    auto I = [&](int k) { return reinterpret_cast<int32_t*>(p + k * i4); };
    auto D = [&](int k) { return reinterpret_cast<double*>(p + 9 * i4 + k * d8); };
    int32_t *best_end = I(0), *exits = I(1), *mark = I(2), *pos = I(3);
    int32_t *st0 = I(4), *st1 = I(5), *en0 = I(6), *en1 = I(7), *gend = I(8);
    double *best_cost = D(0), *cost0 = D(1), *cost1 = D(2), *gcost = D(3);
    SmOpen* open = reinterpret_cast<SmOpen*>(p + 9 * i4 + 4 * d8);
    char* pq = p + 9 * i4 + 4 * d8 + 256;
    i128 *pf1 = reinterpret_cast<i128*>(pq), *pf2 = reinterpret_cast<i128*>(pq + q16);
    i128 *cf1 = reinterpret_cast<i128*>(pq + 2 * q16), *cf2 = reinterpret_cast<i128*>(pq + 2 * q16 + c16);
    char* pt = pq + 2 * q16 + 2 * c16;
    int32_t* tile_tot = reinterpret_cast<int32_t*>(pt);
    int32_t* tile_off = reinterpret_cast<int32_t*>(pt + t4);
    int32_t* entry = reinterpret_cast<int32_t*>(pt + 2 * t4);  // ceil(J / kChain) <= T entries
    static_assert(kChain >= kScanTile, "chain entries fit the scan tiles' array");
    char* ph = pt + 3 * t4;
    const SmHull h{reinterpret_cast<double*>(ph), reinterpret_cast<uint8_t*>(ph + hy),
                   reinterpret_cast<uint8_t*>(ph + hy + hx), slots};
    const SmPrefix pf{pf1, pf2, cf1, cf2, n, JB, B};
    // exclusive scan of mark[0, N) into pos, the total into result[0]
    auto scan_marks = [&](int64_t N) {
        const int64_t nt = (N + kScanTile - 1) / kScanTile;
        hipLaunchKernelGGL(k_sm_scan_local, dim3(static_cast<unsigned>(nt)), dim3(kSmThreads), 0, s, mark, N, pos,
                           tile_tot);
        hipLaunchKernelGGL(k_sm_scan, dim3(1), dim3(kScan), 0, s, tile_tot, nt, tile_off, host.p);
        hipLaunchKernelGGL(k_sm_scan_add, dim3(blocks(N, 256)), dim3(256), 0, s, pos, N, tile_off);
    };
    // the entries that the walk from entry 0 over next() reaches, in order, to
    // emit(entry, position); their number to host.p[0]
    auto chain = [&](auto next, auto emit, int64_t N) {
        using F = decltype(next);
        using E = decltype(emit);
        if (N <= kChain) {
            hipLaunchKernelGGL((k_sm_chain_small<F, E>), dim3(1), dim3(kChainThreads), 0, s, next, emit,
                               static_cast<int32_t>(N), host.p);
            return;
        }
        const unsigned nc = blocks(N, kChain);
        hipLaunchKernelGGL(k_sm_chain_exit<F>, dim3(nc), dim3(kChainThreads), 0, s, next, N, exits);
        hipLaunchKernelGGL(k_sm_chain_walk, dim3(1), dim3(64), 0, s, exits, N, static_cast<int64_t>(nc), entry);
        hipLaunchKernelGGL(k_sm_chain_mark<F>, dim3(nc), dim3(kChainThreads), 0, s, next, N, entry, mark);
        scan_marks(N);
        hipLaunchKernelGGL(k_sm_emit<E>, dim3(blocks(N, 256)), dim3(256), 0, s, mark, pos, N, emit);
    };
    int rc = dispatch_dtype(dtype, [&](auto t) -> int {
        using T = decltype(t);
        const T* v = static_cast<const T*>(d_values);
        if (hulls) {
            hipLaunchKernelGGL(k_sm_blocks<T>, dim3(static_cast<unsigned>(C)), dim3(kBlkThreads), hull_lds(B), s, v, n,
                               B, JB, pf1, pf2, cf1, cf2, h);
        } else {
            hipLaunchKernelGGL(k_sm_sums<T>, dim3(static_cast<unsigned>(JB)), dim3(kSmThreads), 0, s, v, n, B, pf1,
                               pf2);
            hipLaunchKernelGGL(k_sm_chunk_pfx, dim3(static_cast<unsigned>(C)), dim3(kPfxChunk), 0, s, JB, pf1, pf2,
                               cf1, cf2);
        }
        GLC_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_sm_chunk_scan, dim3(1), dim3(kChunkScanThreads), 0, s, cf1, cf2, C);
        if (hulls) {
            hipLaunchKernelGGL(k_sm_split_hull<T>, dim3(blocks(J, split_starts(U))), dim3(kSmThreads),
                               split_lds(U, slots), s, v, n, m, J, U, pf, h, best_end, best_cost);
        } else {
            hipLaunchKernelGGL(k_sm_split<T>, dim3(static_cast<unsigned>(J)), dim3(kSmThreads), 0, s, v, n, m, J,
                               best_end, best_cost);
        }
        GLC_HIP(hipGetLastError());
        chain(ChainSplit{best_end, J, m}, EmitSplit{best_end, best_cost, m, st0, en0, cost0, host.p}, J);
        GLC_HIP(hipGetLastError());
        GLC_HIP(hipStreamSynchronize(s));
        int64_t P = host.p[0];
        if (P < 1 || P > J) return fail(GLC_ERR_STATE, "split phase produced an invalid partition count");
        int32_t *sa = st0, *sb = st1, *ea = en0, *eb = en1;
        double *ca = cost0, *cb = cost1;
        for (int iter = 0; iter < 10 && P > 1; ++iter) {  // CpuPartitioner.cuh:198-242
            const EmitGroups emit{gend, gcost, sa, ea, sb, eb, cb, host.p};
            host.p[2] = 0;  // the stream is idle
            hipLaunchKernelGGL(k_sm_grow<T>, dim3(blocks(P, kSmThreads / 64)), dim3(kSmThreads), 0, s, v, sa, ea, ca,
                               P, pf, h, gend, gcost, host.p + 2);
            chain(ChainMerge{gend}, emit, P);
            GLC_HIP(hipGetLastError());
            GLC_HIP(hipStreamSynchronize(s));
            if (host.p[2]) {  // a group was left open: that list stands only once the walk's are complete
                hipLaunchKernelGGL(k_sm_walk, dim3(1), dim3(kWalkThreads), 0, s, ca, cb, P, true, gend, gcost, open,
                                   host.p + 2);
                while (host.p[2]) {  // each pair ends a group or takes 64 partitions or more into one
                    for (int k = 0; k < 8; ++k) {
                        hipLaunchKernelGGL(k_sm_more<T>, dim3(kMoreCand / (kSmThreads / 64)), dim3(kSmThreads), 0, s, v,
                                           sa, ea, P, pf, h, open, cb);
                        hipLaunchKernelGGL(k_sm_walk, dim3(1), dim3(kWalkThreads), 0, s, ca, cb, P, false, gend, gcost,
                                           open, host.p + 2);
                    }
                    GLC_HIP(hipGetLastError());
                    GLC_HIP(hipStreamSynchronize(s));
                }
                chain(ChainMerge{gend}, emit, P);
                GLC_HIP(hipGetLastError());
                GLC_HIP(hipStreamSynchronize(s));
            }
            const int64_t Pn = host.p[0];
            if (Pn < 1 || Pn > P) return fail(GLC_ERR_STATE, "merge pass produced an invalid partition count");
            const bool changed = Pn < P;  // every merge removes one entry
            P = Pn;
            std::swap(sa, sb);
            std::swap(ea, eb);
            std::swap(ca, cb);
            if (!changed) break;
        }
        out->d_st = sa;
        out->d_en = ea;
        out->P = P;
        out->first_len = host.p[1];
        return GLC_OK;
    });
    if (rc) {
        (void)hipStreamSynchronize(s);  // no kernel of this call may outlive the lock on the scratch
        return rc;
    }
    out->device = dev;
    out->lock = std::move(scratch_lock);
    return GLC_OK;
}

int split_merge_release(SplitMergeResult& r, hipStream_t s) {
    const int rc = scratch_release(sm_scratch(r.device), kSmKeep, s);
    if (!rc) r.lock.unlock();
    return rc;
}

}  // namespace glc
