// glc_decode.hip -- full decompression and pre-unpack kernels of libglc.
//
// Schedules (the reference kernel each mode replaces in parentheses):
//   k_decode_wave       one wave per 1024-element tile, static grid scheduled
//                       by the hardware dispatcher (decompressFullFile_BitPacked /
//                       _PreUnpacked, decompression/FullDecompressionKernels.cuh:48-288,
//                       and decompressFullFile_WorkStealing,
//                       decompression/WorkStealingDecompressionKernels.cuh:332-521)
//   k_decode_plain      pre-unpacked columns of whole-tile partitions, a workgroup per tile
//   k_decode_half       half tiles (GLC_DECODE_HALF_TILE_W1)
//   k_decode_steal      wave tiles claimed from per-XCD atomic queues
//                       (the explicit work-stealing comparator)
// Every full-decode mode takes these.  The reference's per-partition schedules
// (…_OnTheFly_Optimized_V2, FullDecompressionKernels.cuh:293-378, a workgroup
// per partition; …_WorkStealingAdvanced,
// WorkStealingDecompressionKernels.cuh:526-619, workgroups that claim partitions) have no
// kernels of their own: a workgroup per partition was slower than the tiles or within 2 %
// on the layouts measured (tiles / per partition: 2^26 int32 values in partitions of
// 1024, 62 / 105 us; 5e7 int64 in partitions of 64, 100 / 634, of 3000, 75 / 103; 2^27
// int64 pre-unpacked in partitions of 1024, 343 / 358, of 1000, 366 / 372; 5e7 so, into
// an unaligned output, 154 / 152), and claims were slower everywhere (805 and 8913 us on
// the first two).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "glc_device.hpp"
#include "glc_internal.hpp"

namespace glc {
namespace {

enum Op { OP_PACKED = 0, OP_PLAIN = 1, OP_UNPACK = 2 };

struct DecArgs {
    const Desc* __restrict__ desc;
    const int32_t* __restrict__ tile_part;
    const uint32_t* __restrict__ words;
    const int64_t* __restrict__ plain;
    const double* __restrict__ params;   // SoA params (theta2 of POLYNOMIAL2)
    void* __restrict__ out;
    int64_t n;
    int64_t P;
    int64_t n_index;
    const TileInfo* __restrict__ tinfo;  // per-1024-element tile: first bit, bits, partition, path
    int64_t wlimit;                      // payload words (row-load base clamp)
    int32_t* sched;                      // per-XCD work-stealing queues (wave schedule)
    int32_t vec16;                       // out is 16-byte aligned: narrow tiles store 16 bytes per lane
    int32_t skew;                        // values from a 128-byte line's start to out (and to every tile of it)
    bool spans;                          // for the host: some tile holds several partitions (glc_column::spans)
    bool wide;                           // for the host: some field has more than 32 bits
    int32_t pace;                        // pause after each narrow row's stores (pace_row)
    int32_t pace2;                       // the same where predictions are beyond 2^50 (dec_fast_range tier 2)
};

// ---------------------------------------------------------------------------
// Wave-level decoder: no LDS staging and no workgroup barriers.
// A wave owns a 1024-element tile (16 rows of 64 elements).  The tile's
// TileInfo (first bit, bit width, partition, path) is one 16-byte load.  For
// each row the wave issues one fully coalesced dword load of the row's words
// (lane l loads word l); all 16 row loads are issued before any compute, so
// the wave never waits on its own stores (vmcnt is in-order on gfx9).  Each
// lane then picks the 2-3 words its element needs with ds_bpermute, extracts
// the field with v_alignbit_b32 + v_bfe_i32, and stores with a non-temporal
// store (64 consecutive elements per row: fully coalesced).
// ---------------------------------------------------------------------------
constexpr int kWaveRows = 16;
constexpr int kWaveTile = 64 * kWaveRows;  // == kIndexTile: a wave tile starts on an index entry
constexpr int kWavesPerGroup = 4;
static_assert(kWaveTile == kIndexTile, "wave tiles are aligned to the partition index");

__device__ __forceinline__ uint32_t bperm(uint32_t v, uint32_t src_lane) {
    return static_cast<uint32_t>(
        __builtin_amdgcn_ds_bpermute(static_cast<int>((src_lane & 63u) << 2), static_cast<int>(v)));
}

template <class V> __device__ __forceinline__ void put(V* p, V v) { __builtin_nontemporal_store(v, p); }

template <class T, int OP>
__device__ __forceinline__ void emit(const DecArgs& a, int64_t e, int32_t type, double t0, double t1, int32_t i,
                                     uint64_t raw, int64_t delta) {
    if constexpr (OP == OP_UNPACK) {
        put(static_cast<int64_t*>(a.out) + e,
            (type == MODEL_DIRECT_COPY) ? static_cast<int64_t>(static_cast<T>(raw)) : delta);
    } else {
        put(static_cast<T*>(a.out) + e, (type == MODEL_DIRECT_COPY) ? static_cast<T>(raw)
                                                                    : apply_delta<T>(dec_pred<T>(t0, t1, i), delta));
    }
}

// Rows of a tile whose output is not 16-byte aligned: row 0 ends at a line of the
// output, the others are 64 values from there on, so that only a tile's two ends
// share a line with another wave's stores (5e7 int64 values in partitions of 64: 134
// us with rows across lines, 103 so).  SKEW = false: plain rows of 64.
constexpr int kSkewRows = kWaveRows + 1;
template <bool SKEW> __device__ __forceinline__ int32_t row_start(int r, int32_t skew) {
    return SKEW && r > 0 ? r * 64 - skew : r * 64;
}
template <bool SKEW> __device__ __forceinline__ int32_t row_end(int r, int32_t skew) {
    return SKEW ? (r + 1) * 64 - skew : (r + 1) * 64;
}

// Index in the partition of the tile's value k; past the tile's end (k up to 1087,
// never stored) it may wrap.
__device__ __forceinline__ int32_t local_of(const TileInfo& x, int32_t k) {
    return static_cast<int32_t>(static_cast<uint32_t>(x.lbase) + static_cast<uint32_t>(k));
}

// Narrow fast path, outputs that are not 16-byte aligned: the tile lies in one
// partition with bits <= 32 (linear model).  FAST as in narrow_v_rows.
template <class T, int FAST>
__device__ __forceinline__ void narrow_rows(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                            const uint32_t (&x0)[kSkewRows], const uint32_t (&xs)[kSkewRows]) {
    const int b = tile_bits(x.info);
    const uint32_t rel_lane = static_cast<uint32_t>(lane) * static_cast<uint32_t>(b);
    T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
    for (int r = 0; r < kSkewRows; ++r) {
        const int32_t k = row_start<true>(r, a.skew) + lane;
        const int64_t R = x.W + static_cast<int64_t>(row_start<true>(r, a.skew)) * b;
        const uint32_t rel = static_cast<uint32_t>(R & 31) + rel_lane;
        const uint32_t wi = rel >> 5;
        const uint32_t lo = bperm(x0[r], wi);
        const uint32_t hb = bperm(x0[r], wi + 1);
        const uint32_t hi = (wi + 1 < 64) ? hb : xs[r];
        const uint32_t raw = __builtin_amdgcn_alignbit(hi, lo, rel & 31);
        // the builtin returns an unsigned: sign-extend through int32
        const int64_t delta = b == 32 ? static_cast<int64_t>(static_cast<int32_t>(raw))
                                      : static_cast<int64_t>(static_cast<int32_t>(__builtin_amdgcn_sbfe(
                                            static_cast<int>(raw), 0u, static_cast<unsigned>(b))));
        T v;
        const int32_t i = local_of(x, k);
        if constexpr (FAST != 0) v = apply_delta<T>(dec_pred_fast<T, FAST>(x.t0, x.t1, i), delta);
        else v = apply_delta<T>(dec_pred<T>(x.t0, x.t1, i), delta);
        if (k < row_end<true>(r, a.skew) && e0 + k < e1) put(out + e0 + k, v);
    }
}

template <class T, int TIER = 1> __device__ __forceinline__ bool tile_fast(const TileInfo& x, int32_t i0, int32_t i1);

template <class T>
__device__ __forceinline__ void wave_narrow(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane) {
    const int b = tile_bits(x.info);
    const uint32_t* __restrict__ w = a.words;
    uint32_t x0[kSkewRows], xs[kSkewRows];
    // Branch-free loads: lane l reads word wb + l of the row, plus word wb + 64.
    // wb is clamped to the payload end (rows past the column end are never
    // stored), and the payload carries kPayloadPadWords zero words, so every
    // read stays inside the allocation.
#pragma unroll
    for (int r = 0; r < kSkewRows; ++r) {
        const int64_t R = x.W + static_cast<int64_t>(row_start<true>(r, a.skew)) * b;
        const int64_t wb = (R >> 5) < a.wlimit ? (R >> 5) : a.wlimit;
        x0[r] = w[wb + lane];
        xs[r] = w[wb + 64];
    }
    if (tile_fast<T, 1>(x, x.lbase, x.lbase + kWaveTile - 1)) narrow_rows<T, 1>(a, x, e0, e1, lane, x0, xs);
    else narrow_rows<T, 0>(a, x, e0, e1, lane, x0, xs);
}

// Narrow path with V adjacent values per lane and one 16-byte store per lane
// and row (8 bytes when V * sizeof(output) is 8): a row is 64*V values, a
// tile 1024/(64*V) rows.  Needs V * bits <= 64, so a lane's field starts in
// one of its first two words and the lane's V fields span at most three
// words of the row window (words wb .. wb+128, as wave_narrow's rows).
// Fewer, wider stores per wave: 8 instead of 16 for 64-bit values, 4
// instead of 16 for 32-bit values with fields of at most 16 bits.
// NP = 1: the whole tile; NP = 2: half h of the tile's rows (the half-tile
// schedule, one wave per half): rows rbase ...
// Pause after a row's stores: the column's decode pace, in units of 64
// cycles (0 = none).  Less arithmetic between a wave's stores made some
// decodes slower; a pause restores the spacing.  On the 4 GiB int64
// timestamp column the half-tile decode ran 0.945 ms back to back with no
// pause and 0.88-0.90 ms with 16 per row (32: 1.00 ms); the uint64 2^28
// column and the int32 column are fastest without.  The autotuner picks it
// with the schedule.
__device__ __forceinline__ void pace_row(int32_t pace) {
    if (pace == 4) __builtin_amdgcn_s_sleep(4);
    else if (pace == 8) __builtin_amdgcn_s_sleep(8);
    else if (pace == 16) __builtin_amdgcn_s_sleep(16);
    else if (pace == 24) __builtin_amdgcn_s_sleep(24);
}

// FAST: 0 = the saturating conversion (dec_pred); 1 or 2 = every prediction
// of the wave's rows lies in dec_fast_range of that tier; FULL: every row
// lies inside the column (no per-row end check).
template <class T, int OP, int V, int FAST, bool FULL, int NR>
__device__ __forceinline__ void narrow_v_rows(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                              int rbase, const uint32_t (&x0)[NR], const uint32_t (&x1)[NR],
                                              const uint32_t (&xs)[NR]) {
    typedef typename std::conditional<OP == OP_UNPACK, int64_t, T>::type O;  // output element
    constexpr int kRowVals = 64 * V;
    const int b = tile_bits(x.info);
    const int32_t lbase = x.lbase;
    const uint32_t rel_lane = static_cast<uint32_t>(lane) * static_cast<uint32_t>(V * b);
    O* __restrict__ out = static_cast<O*>(a.out);
#pragma unroll
    for (int rr = 0; rr < NR; ++rr) {
        const int r = rbase + rr;
        const int64_t R = x.W + static_cast<int64_t>(r * kRowVals) * b;
        const uint32_t rel = static_cast<uint32_t>(R & 31) + rel_lane;
        const uint32_t wi = rel >> 5, sh = rel & 31;
        uint32_t g[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {  // words wi .. wi+2 of the row window (wi + 2 <= 128)
            const uint32_t j = wi + k;
            const uint32_t p0 = bperm(x0[rr], j), p1 = bperm(x1[rr], j);
            g[k] = (j < 64) ? p0 : (j < 128) ? p1 : xs[rr];
        }
        O v[V];
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const uint32_t sk = sh + k * b;  // < 96; a field starting at bit 64 or later ends inside g[2]
            const uint32_t idx = sk >> 5;
            const uint32_t lo = idx == 0 ? g[0] : idx == 1 ? g[1] : g[2];
            const uint32_t hi = idx == 0 ? g[1] : g[2];
            const uint32_t raw = __builtin_amdgcn_alignbit(hi, lo, sk & 31);
            // the builtin returns an unsigned: sign-extend through int32
            const int64_t delta = (b == 32) ? static_cast<int64_t>(static_cast<int32_t>(raw))
                                            : static_cast<int64_t>(static_cast<int32_t>(__builtin_amdgcn_sbfe(
                                                  static_cast<int>(raw), 0u, static_cast<unsigned>(b))));
            const int32_t i = lbase + r * kRowVals + lane * V + k;
            if constexpr (OP == OP_UNPACK) v[k] = delta;
            else if constexpr (FAST != 0) v[k] = apply_delta<T>(dec_pred_fast<T, FAST>(x.t0, x.t1, i), delta);
            else v[k] = apply_delta<T>(dec_pred<T>(x.t0, x.t1, i), delta);
        }
        const int64_t e = e0 + r * kRowVals + lane * V;
        if (FULL || e + V <= e1) {
            if constexpr (V * sizeof(O) == 16) {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                u32x4 q;
                if constexpr (sizeof(O) == 8) {
                    q.x = static_cast<uint32_t>(static_cast<uint64_t>(v[0]));
                    q.y = static_cast<uint32_t>(static_cast<uint64_t>(v[0]) >> 32);
                    q.z = static_cast<uint32_t>(static_cast<uint64_t>(v[1]));
                    q.w = static_cast<uint32_t>(static_cast<uint64_t>(v[1]) >> 32);
                } else {
                    q.x = static_cast<uint32_t>(v[0]);
                    q.y = static_cast<uint32_t>(v[1]);
                    q.z = static_cast<uint32_t>(v[2]);
                    q.w = static_cast<uint32_t>(v[3]);
                }
                put(reinterpret_cast<u32x4*>(out + e), q);
            } else {
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                u32x2 q;
                q.x = static_cast<uint32_t>(v[0]);
                q.y = static_cast<uint32_t>(v[1]);
                put(reinterpret_cast<u32x2*>(out + e), q);
            }
        } else {
#pragma unroll
            for (int k = 0; k < V; ++k)
                if (e + k < e1) put(out + e + k, v[k]);
        }
        if constexpr (FAST == 1) pace_row(a.pace);
        else if constexpr (FAST == 2) pace_row(a.pace2);
    }
}

// True when every prediction of local indices i0 .. i1 of the tile's
// partition lies in dec_fast_range<T, TIER> (the same on every lane).
template <class T, int TIER>
__device__ __forceinline__ bool tile_fast(const TileInfo& x, int32_t i0, int32_t i1) {
    const bool f = dec_fast_range<T, TIER>(__builtin_fma(x.t1, static_cast<double>(i0), x.t0),
                                           __builtin_fma(x.t1, static_cast<double>(i1), x.t0));
    return __builtin_amdgcn_readfirstlane(static_cast<int>(f)) != 0;
}

template <class T, int OP>
__device__ __forceinline__ void wave_slow(const DecArgs& a, int64_t e0, int64_t e1, int64_t plo, int lane);

template <class T, int OP, int V, int NP = 1>
__device__ __forceinline__ void wave_narrow_v(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                              int h = 0) {
    constexpr int kRowVals = 64 * V;
    constexpr int kRows = kWaveTile / kRowVals / NP;
    static_assert(kRows >= 1, "a part holds at least one row");
    static_assert(V * sizeof(typename std::conditional<OP == OP_UNPACK, int64_t, T>::type) == 16 ||
                      V * sizeof(typename std::conditional<OP == OP_UNPACK, int64_t, T>::type) == 8,
                  "16- or 8-byte stores");
    const int rbase = h * kRows;
    const int b = tile_bits(x.info);
    const uint32_t* __restrict__ w = a.words;
    uint32_t x0[kRows], x1[kRows], xs[kRows];
    // Branch-free loads of the 129-word row window (wb clamped as in
    // wave_narrow).  Lanes whose word lies past the last word of the wave's
    // fields (wend) load word wend instead: such words are never selected by
    // a field, and the wave then touches no cache line of the next wave's
    // range (which another XCD may be reading) -- 1-2 % faster than the full
    // window, while exec-masked loads of only the spanned words ran 5-10 %
    // slower.
    const int64_t wend = (x.W + static_cast<int64_t>((rbase + kRows) * kRowVals) * b - 1) >> 5;
#pragma unroll
    for (int rr = 0; rr < kRows; ++rr) {
        const int r = rbase + rr;
        const int64_t R = x.W + static_cast<int64_t>(r * kRowVals) * b;
        const int64_t wb = (R >> 5) < a.wlimit ? (R >> 5) : a.wlimit;
        const int64_t d = wend - wb;
        const uint32_t lim = static_cast<uint32_t>(d < 0 ? 0 : d > 128 ? 128 : d);
        const uint32_t l0 = static_cast<uint32_t>(lane) < lim ? static_cast<uint32_t>(lane) : lim;
        const uint32_t l1 = static_cast<uint32_t>(64 + lane) < lim ? static_cast<uint32_t>(64 + lane) : lim;
        x0[rr] = w[wb + l0];
        x1[rr] = w[wb + l1];
        xs[rr] = w[wb + lim];
    }
    if constexpr (OP == OP_PACKED) {
        const int32_t i0 = x.lbase + rbase * kRowVals;
        const int32_t i1 = i0 + kRows * kRowVals - 1;
        const bool full = e0 + (rbase + kRows) * kRowVals <= e1;
        if (tile_fast<T, 1>(x, i0, i1)) {
            if (full) narrow_v_rows<T, OP, V, 1, true>(a, x, e0, e1, lane, rbase, x0, x1, xs);
            else narrow_v_rows<T, OP, V, 1, false>(a, x, e0, e1, lane, rbase, x0, x1, xs);
            return;
        }
        if constexpr (sizeof(T) == 8) {  // 64-bit predictions beyond 2^50 (timestamps, large offsets)
            if (tile_fast<T, 2>(x, i0, i1)) {
                if (full) narrow_v_rows<T, OP, V, 2, true>(a, x, e0, e1, lane, rbase, x0, x1, xs);
                else narrow_v_rows<T, OP, V, 2, false>(a, x, e0, e1, lane, rbase, x0, x1, xs);
                return;
            }
        }
        // predictions that saturate (beyond T, NaN): the general per-lane path
        // over this wave's rows.  Carrying the saturating conversion through
        // the unrolled rows instead cost ~8 KB of code per element type for a
        // case only extreme fits reach.
        const int64_t p0 = e0 + rbase * kRowVals;
        const int64_t p1 = (e0 + (rbase + kRows) * kRowVals < e1) ? e0 + (rbase + kRows) * kRowVals : e1;
        wave_slow<T, OP>(a, p0, p1, a.tile_part[e0 >> kIndexShift], lane);
    } else {
        narrow_v_rows<T, OP, V, 0, false>(a, x, e0, e1, lane, rbase, x0, x1, xs);
    }
}

// Wide fast path: one partition, 33..64-bit fields or DIRECT_COPY; two row
// registers per row (words l and 64 + l) and three bpermute pairs per element.
// NP, h: part h of NP of the tile's rows.
template <class T, int OP, int NP = 1>
__device__ __forceinline__ void wave_wide(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                          int h = 0) {
    constexpr int kRows = kWaveRows / NP;
    static_assert(kRows % 4 == 0, "whole groups of rows");
    const int b = tile_bits(x.info);
    const uint32_t* __restrict__ w = a.words;
    const int32_t type = tile_type(x.info);
    const uint32_t rel_lane = static_cast<uint32_t>(lane) * static_cast<uint32_t>(b);
    for (int r0 = h * kRows; r0 < (h + 1) * kRows; r0 += 4) {
        uint32_t x0[4], x1[4], xs[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {  // branch-free, clamped as in wave_narrow
            const int64_t R = x.W + static_cast<int64_t>((r0 + k) * 64) * b;
            const int64_t wb = (R >> 5) < a.wlimit ? (R >> 5) : a.wlimit;
            x0[k] = w[wb + lane];
            x1[k] = w[wb + 64 + lane];
            xs[k] = w[wb + 128];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t e = e0 + (r0 + k) * 64 + lane;
            const int64_t R = x.W + static_cast<int64_t>((r0 + k) * 64) * b;
            const uint32_t rel = static_cast<uint32_t>(R & 31) + rel_lane;
            const uint32_t wi = rel >> 5;
            const uint32_t w1 = wi + 1, w2 = wi + 2;
            const uint32_t l0 = bperm(x0[k], wi), l1 = bperm(x1[k], wi);
            const uint32_t a0 = bperm(x0[k], w1), a1 = bperm(x1[k], w1);
            const uint32_t c0 = bperm(x0[k], w2), c1 = bperm(x1[k], w2);
            const uint32_t lo = (wi < 64) ? l0 : l1;
            const uint32_t hi = (w1 < 64) ? a0 : a1;
            const uint32_t top = (w2 < 64) ? c0 : (w2 < 128) ? c1 : xs[k];
            const uint32_t s = rel & 31;
            const uint64_t raw = (static_cast<uint64_t>(__builtin_amdgcn_alignbit(top, hi, s)) << 32) |
                                 __builtin_amdgcn_alignbit(hi, lo, s);
            const uint64_t rawv = (b >= 64) ? raw : (raw & ((1ULL << b) - 1ULL));
            const int64_t delta =
                (b >= 64) ? static_cast<int64_t>(raw) : static_cast<int64_t>(raw << (64 - b)) >> (64 - b);
            if (e < e1) emit<T, OP>(a, e, type, x.t0, x.t1, x.lbase + (r0 + k) * 64 + lane, rawv, delta);
        }
    }
}

// V adjacent values of a lane at p: those with index in [lo, hi) of them, one
// 16- or 8-byte store when that is all (p is aligned to it).
template <class O, int V>
__device__ __forceinline__ void put_values(O* p, const O (&v)[V], int32_t lo, int32_t hi) {
    if (lo <= 0 && hi >= V) {
        if constexpr (V * sizeof(O) == 16) {
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            u32x4 q;
            if constexpr (sizeof(O) == 8) {
                q.x = static_cast<uint32_t>(static_cast<uint64_t>(v[0]));
                q.y = static_cast<uint32_t>(static_cast<uint64_t>(v[0]) >> 32);
                q.z = static_cast<uint32_t>(static_cast<uint64_t>(v[1]));
                q.w = static_cast<uint32_t>(static_cast<uint64_t>(v[1]) >> 32);
            } else {
                q.x = static_cast<uint32_t>(v[0]);
                q.y = static_cast<uint32_t>(v[1]);
                q.z = static_cast<uint32_t>(v[2]);
                q.w = static_cast<uint32_t>(v[3]);
            }
            put(reinterpret_cast<u32x4*>(p), q);
        } else if constexpr (V == 2) {
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            u32x2 q;
            q.x = static_cast<uint32_t>(v[0]);
            q.y = static_cast<uint32_t>(v[1]);
            put(reinterpret_cast<u32x2*>(p), q);
        } else {
            put(p, v[0]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < V; ++k)
            if (k >= lo && k < hi) put(p + k, v[k]);
    }
}

// Pre-unpacked deltas, two per lane: one 16-byte load of two adjacent int64
// deltas and one 16-byte (8-byte for 32-bit values) store per lane and row
// of 128 values.  SKEW: the output is not 16-byte aligned; row r starts at tile
// value 128 r - skew, on a line of it, so that the stores are aligned all the same and
// the deltas' loads to 8 bytes (1e8 int64 values: a value a lane in rows of 64 across
// lines 381 us, 265 so).  PRED: 0 = DIRECT_COPY, 1 = dec_pred,
// 2 / 3 = dec_pred_fast of tier 1 / 2.
typedef int64_t i64x2 __attribute__((ext_vector_type(2), aligned(8)));
constexpr int kPlainRows = kWaveTile / 128;

template <class T, int PRED, int NR, bool SKEW>
__device__ __forceinline__ void plain_v_rows(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                             int rbase, const i64x2 (&pl)[NR]) {
    T* __restrict__ out = static_cast<T*>(a.out);
    const int32_t cnt = static_cast<int32_t>(e1 - e0);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int32_t k = (rbase + r) * 128 + 2 * lane - (SKEW ? a.skew : 0);
        const int32_t i = local_of(x, k);
        T v[2];
        if constexpr (PRED == 0) {
            v[0] = static_cast<T>(pl[r].x);
            v[1] = static_cast<T>(pl[r].y);
        } else if constexpr (PRED == 1) {
            v[0] = apply_delta<T>(dec_pred<T>(x.t0, x.t1, i), pl[r].x);
            v[1] = apply_delta<T>(dec_pred<T>(x.t0, x.t1, local_of(x, k + 1)), pl[r].y);
        } else {
            v[0] = apply_delta<T>(dec_pred_fast<T, PRED - 1>(x.t0, x.t1, i), pl[r].x);
            v[1] = apply_delta<T>(dec_pred_fast<T, PRED - 1>(x.t0, x.t1, local_of(x, k + 1)), pl[r].y);
        }
        put_values<T, 2>(out + e0 + k, v, SKEW ? -k : 0, cnt - k);
    }
}

// NP, h: part h of NP of the tile's rows (SKEW: the last part's with what row 0
// leaves over).
template <class T, int NP = 1, bool SKEW = false>
__device__ __forceinline__ void wave_plain_v(const DecArgs& a, const TileInfo& x, int64_t e0, int64_t e1, int lane,
                                             int h = 0) {
    constexpr int kRows = kPlainRows / NP + (SKEW ? 1 : 0);
    const int rbase = h * (kPlainRows / NP);
    // values of this part
    const int64_t end = SKEW && h < NP - 1 ? e0 + (rbase + kRows - 1) * 128 - a.skew : e1;
    const int32_t cnt = static_cast<int32_t>((end < e1 ? end : e1) - e0);
    i64x2 pl[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int32_t k = (rbase + r) * 128 + 2 * lane - (SKEW ? a.skew : 0);
        if (k >= 0 && k + 2 <= cnt) {
            pl[r] = *reinterpret_cast<const i64x2*>(a.plain + e0 + k);
        } else {
            pl[r].x = (k >= 0 && k < cnt) ? a.plain[e0 + k] : 0;
            pl[r].y = (k + 1 >= 0 && k + 1 < cnt) ? a.plain[e0 + k + 1] : 0;
        }
    }
    const int64_t stop = e0 + cnt;
    if (tile_type(x.info) == MODEL_DIRECT_COPY) plain_v_rows<T, 0, kRows, SKEW>(a, x, e0, stop, lane, rbase, pl);
    else if (tile_fast<T, 1>(x, x.lbase, x.lbase + kWaveTile - 1))
        plain_v_rows<T, 2, kRows, SKEW>(a, x, e0, stop, lane, rbase, pl);
    else if (sizeof(T) == 8 && tile_fast<T, 2>(x, x.lbase, x.lbase + kWaveTile - 1))
        plain_v_rows<T, 3, kRows, SKEW>(a, x, e0, stop, lane, rbase, pl);
    else plain_v_rows<T, 1, kRows, SKEW>(a, x, e0, stop, lane, rbase, pl);
}

// Slow path: a tile spanning several partitions, gaps, or a decode-only
// polynomial model.  Per-lane partition search inside the tile's candidate
// range, direct extraction from global memory.
template <class T, int OP>
__device__ __forceinline__ void wave_slow(const DecArgs& a, int64_t e0, int64_t e1, int64_t plo, int lane) {
    const int64_t phi = a.tile_part[(e1 + kIndexTile - 1) >> kIndexShift];
    for (int64_t e = e0 + lane; e < e1; e += 64) {
        int64_t lo = plo, hi = phi;
        while (lo < hi) {
            const int64_t m = (lo + hi + 1) >> 1;
            if (a.desc[m].start <= e) lo = m; else hi = m - 1;
        }
        const Desc d = a.desc[lo];
        const int64_t k = e - d.start;
        if (k < 0 || k >= d.len) {
            if constexpr (OP == OP_UNPACK) static_cast<int64_t*>(a.out)[e] = 0;
            else static_cast<T*>(a.out)[e] = T(0);
            continue;
        }
        const int32_t type = desc_type(d.packed);
        const int b = desc_bits(d.packed);
        const int32_t i = static_cast<int32_t>(k);
        if constexpr (OP == OP_PLAIN) {
            const int64_t pl = a.plain[e];
            T v;
            if (type == MODEL_DIRECT_COPY) v = static_cast<T>(pl);
            else if (type == MODEL_POLY2)
                v = apply_delta<T>(dec_pred_poly<T>(type, d.theta0, d.theta1, a.params[4 * lo + 2], i), pl);
            else v = apply_delta<T>(dec_pred<T>(d.theta0, d.theta1, i), pl);
            static_cast<T*>(a.out)[e] = v;
        } else {
            const uint64_t raw = (b > 0) ? extract_raw_g(a.words, desc_off(d.packed) + k * b, b) : 0;
            const int64_t delta = sign_extend(raw, b);
            if (OP == OP_PACKED && type == MODEL_POLY2) {
                static_cast<T*>(a.out)[e] =
                    apply_delta<T>(dec_pred_poly<T>(type, d.theta0, d.theta1, a.params[4 * lo + 2], i), delta);
            } else {
                emit<T, OP>(a, e, type, d.theta0, d.theta1, i, raw, delta);
            }
        }
    }
}

// Tiles that hold several partitions (or a gap, or a decode-only polynomial
// model), kSegParts at most: partition by partition, the whole wave on one at a
// time, so that the model and the bit width are wave-uniform and neighbouring
// lanes read neighbouring words.  Lanes take V adjacent values aligned to V in
// the tile (one 16-byte store where all of them are the partition's), V fields
// of V * bits <= 64 from three words loaded together, or two wider ones from five.
// The next partition's descriptor is loaded before the current one is decoded.
// 5e7 uint32 values in partitions of 1000: 57 us, where a search per value
// (wave_slow) took 225 us and wave_many takes 90; from about 300 values a partition
// down wave_many is the faster one (300: 81 against 134 us).  Bound by the work per
// row: rows past the partition are left out (64 us with them), and one of two
// wide fields a lane costs 4/5 of two rows of one (7e7 uint64, 36 bits, S = 1000:
// 208 -> 160 us).
constexpr int kSegParts = 3;

// Values [s, t) of partition p (descriptor d; s, t in elements) of the tile at
// e0.  FAST as in narrow_v_rows; 0 also takes DIRECT_COPY and POLY2.  WIDE: two
// fields of up to 64 bits from five words.
template <class T, int OP, int V, int FAST, bool WIDE = false, bool VEC = true>
__device__ __forceinline__ void seg_rows(const DecArgs& a, const Desc& d, int64_t p, int64_t e0, int64_t s, int64_t t,
                                         int lane) {
    typedef typename std::conditional<OP == OP_UNPACK, int64_t, T>::type O;
    // in flight; more only cost registers (V = 1 with 8: 128 against 117 us; V = 2
    // and 4 with as many as a tile has: 2 to 60 % slower)
    constexpr int kSegRows = V == 4 ? 2 : 4;
    constexpr int kWords = WIDE ? 5 : 3;
    static_assert(!WIDE || V == 2, "two wide fields");
    O* __restrict__ out = static_cast<O*>(a.out);
    const int b = desc_bits(d.packed);
    const int32_t type = desc_type(d.packed);
    const int64_t off = desc_off(d.packed);
    const double t2 = (FAST == 0 && OP != OP_UNPACK && type == MODEL_POLY2) ? a.params[4 * p + 2] : 0.0;
    const int32_t lo = static_cast<int32_t>(s - e0), hi = static_cast<int32_t>(t - e0);  // in the tile
    const int32_t kb = static_cast<int32_t>(e0 - d.start);  // tile position x is value kb + x of the partition
    constexpr int32_t kLine = 128 / sizeof(O);  // rows on whole lines (partitions of 1000: 1-4 %)
    const int32_t skew = VEC ? 0 : a.skew;
    for (int32_t row = (lo + skew) / kLine * kLine - skew; row < hi; row += kSegRows * 64 * V) {
        const int32_t x0 = row + lane * V;
        uint32_t w[kSegRows][kWords];
        int64_t pl[kSegRows][V];
#pragma unroll
        for (int r = 0; r < kSegRows; ++r) {
            const int32_t x = x0 + r * 64 * V;
            if (r > 0 && row + r * 64 * V >= hi) continue;
            if constexpr (OP == OP_PLAIN) {
#pragma unroll
                for (int j = 0; j < V; ++j) pl[r][j] = a.plain[e0 + (x + j < lo ? lo : x + j < hi ? x + j : hi - 1)];
            } else {  // the words from the lane's first field of the partition on
                const int32_t xf = x < lo ? lo : x < hi ? x : hi - 1;
                const int64_t wi = (off + static_cast<int64_t>(kb + xf) * b) >> 5;
#pragma unroll
                for (int q = 0; q < kWords; ++q) w[r][q] = a.words[wi + q];
            }
        }
#pragma unroll
        for (int r = 0; r < kSegRows; ++r) {
            const int32_t x = x0 + r * 64 * V;
            if (r > 0 && row + r * 64 * V >= hi) continue;
            const int32_t xf = x < lo ? lo : x < hi ? x : hi - 1;
            const uint32_t sh = static_cast<uint32_t>(off + static_cast<int64_t>(kb + xf) * b) & 31;
            O v[V];
#pragma unroll
            for (int j = 0; j < V; ++j) {
                uint64_t raw;
                int64_t delta;
                if constexpr (OP == OP_PLAIN) {
                    delta = pl[r][j];
                    raw = static_cast<uint64_t>(delta);
                } else if constexpr (V == 1) {
                    raw = static_cast<uint64_t>(__builtin_amdgcn_alignbit(w[r][2], w[r][1], sh)) << 32 |
                          __builtin_amdgcn_alignbit(w[r][1], w[r][0], sh);
                    delta = sign_extend(raw, b);
                    raw = b >= 64 ? raw : raw & ((1ULL << b) - 1ULL);
                } else if constexpr (WIDE) {
                    const uint32_t sk = sh + (x + j > xf ? static_cast<uint32_t>(b) : 0u);  // second field: 33 .. 95
                    const uint32_t idx = sk >> 5;
                    const uint32_t l = idx == 0 ? w[r][0] : idx == 1 ? w[r][1] : w[r][2];
                    const uint32_t m = idx == 0 ? w[r][1] : idx == 1 ? w[r][2] : w[r][3];
                    const uint32_t h = idx == 0 ? w[r][2] : idx == 1 ? w[r][3] : w[r][4];
                    raw = static_cast<uint64_t>(__builtin_amdgcn_alignbit(h, m, sk & 31)) << 32 |
                          __builtin_amdgcn_alignbit(m, l, sk & 31);
                    delta = sign_extend(raw, b);
                    raw = b >= 64 ? raw : raw & ((1ULL << b) - 1ULL);
                } else {
                    const int32_t jj = x + j - xf;  // fields after the first loaded one
                    const uint32_t sk = sh + static_cast<uint32_t>(jj < 0 ? 0 : jj) * b;
                    const uint32_t idx = sk >> 5;
                    const uint32_t l = idx == 0 ? w[r][0] : idx == 1 ? w[r][1] : w[r][2];
                    const uint32_t h = idx == 0 ? w[r][1] : w[r][2];
                    const uint32_t f = __builtin_amdgcn_alignbit(h, l, sk & 31);
                    raw = b == 32 ? f : f & ((1u << b) - 1u);
                    // the builtin returns an unsigned: sign-extend through int32
                    delta = b == 32 ? static_cast<int64_t>(static_cast<int32_t>(f))
                                    : static_cast<int64_t>(static_cast<int32_t>(__builtin_amdgcn_sbfe(
                                          static_cast<int>(f), 0u, static_cast<unsigned>(b))));
                }
                const int32_t i = kb + x + j;
                if constexpr (FAST != 0) v[j] = apply_delta<T>(dec_pred_fast<T, FAST>(d.theta0, d.theta1, i), delta);
                else if constexpr (OP == OP_UNPACK)
                    v[j] = type == MODEL_DIRECT_COPY ? static_cast<int64_t>(static_cast<T>(raw)) : delta;
                else
                    v[j] = type == MODEL_DIRECT_COPY
                               ? static_cast<T>(raw)
                               : apply_delta<T>(dec_pred_poly<T>(type, d.theta0, d.theta1, t2, i), delta);
            }
            put_values<O, V>(out + e0 + x, v, lo - x, hi - x);
        }
    }
}

// Values [s, t) of one partition of the tile at e0 (wave-uniform arguments).
template <class T, int OP, bool VEC>
__device__ __forceinline__ void seg_decode(const DecArgs& a, const Desc& d, int64_t p, int64_t e0, int64_t s,
                                           int64_t t, int lane) {
    constexpr int kWide = (OP == OP_UNPACK || sizeof(T) == 8) ? 2 : 4;  // values of a 16-byte store
    const int b = desc_bits(d.packed);
    const int32_t type = desc_type(d.packed);
    if constexpr (OP == OP_PACKED) {
        const double p0 = __builtin_fma(d.theta1, static_cast<double>(s - d.start), d.theta0);
        const double p1 = __builtin_fma(d.theta1, static_cast<double>(t - 1 - d.start), d.theta0);
        const bool line = type != MODEL_DIRECT_COPY && type != MODEL_POLY2;
        const int tier = !line ? 0 : dec_fast_range<T, 1>(p0, p1) ? 1 : (sizeof(T) == 8 && dec_fast_range<T, 2>(p0, p1)) ? 2 : 0;
        const int u = __builtin_amdgcn_readfirstlane(tier);
        if (b <= 64 / kWide && b <= 32) {
            if (u == 1) seg_rows<T, OP, kWide, 1, false, VEC>(a, d, p, e0, s, t, lane);
            else if (sizeof(T) == 8 && u == 2) seg_rows<T, OP, kWide, 2, false, VEC>(a, d, p, e0, s, t, lane);
            else seg_rows<T, OP, 1, 0, false, VEC>(a, d, p, e0, s, t, lane);
        } else if (sizeof(T) == 4 && b <= 32 && u == 1) {
            seg_rows<T, OP, 2, 1, false, VEC>(a, d, p, e0, s, t, lane);
        } else if constexpr (sizeof(T) == 8) {
            if (u == 1) seg_rows<T, OP, 2, 1, true, VEC>(a, d, p, e0, s, t, lane);
            else if (u == 2) seg_rows<T, OP, 2, 2, true, VEC>(a, d, p, e0, s, t, lane);
            else seg_rows<T, OP, 1, 0, false, VEC>(a, d, p, e0, s, t, lane);
        } else {
            seg_rows<T, OP, 1, 0, false, VEC>(a, d, p, e0, s, t, lane);
        }
    } else if constexpr (OP == OP_UNPACK) {
        if (b <= 32) seg_rows<T, OP, 2, 0>(a, d, p, e0, s, t, lane);
        else seg_rows<T, OP, 2, 0, true>(a, d, p, e0, s, t, lane);
    } else {
        seg_rows<T, OP, 2, 0, false, VEC>(a, d, p, e0, s, t, lane);
    }
}

// Tiles of more than kSegParts partitions, a value per lane: the staged
// partition map (ManyLds) instead of a search, the payload loads of four rows in
// flight together.  5e7 values in partitions of 64: 83-121 us by type and width
// where the search took 300-350.  Returns false (nothing written) where the map
// does not apply: the caller searches.
//
// The staged form: value x of the tile is the partition's value x - sx and its
// first bit is bit off + x * bits of the payload.
struct alignas(8) ManyDesc {
    double t0, t1;
    int64_t off;
    int32_t sx;
    uint32_t len;
    int32_t info;  // bits | type << 8 | tier << 12 (dec_fast_range over the whole partition, 0 = none)
    int32_t pad;
};
struct ManyLds {
    ManyDesc d[kManyParts];
    uint32_t bits[kManyBits];
};

template <class T, int OP, bool SKEW>
__device__ __forceinline__ bool wave_many(const DecArgs& a, int64_t e0, int64_t e1, int64_t plo, int np, int lane,
                                          ManyLds& L) {
    typedef typename std::conditional<OP == OP_UNPACK, int64_t, T>::type O;
    O* __restrict__ out = static_cast<O*>(a.out) + e0;
    int wide = 0;
    const bool ok = many_stage(plo, np, lane, L.bits, [&](int64_t p, int i) {
        const Desc d = a.desc[p];
        const int b = desc_bits(d.packed), type = desc_type(d.packed);
        const int32_t sx = static_cast<int32_t>(d.start - e0);
        int tier = 0;
        if (OP != OP_UNPACK && type != MODEL_DIRECT_COPY && type != MODEL_POLY2 && d.len > 0) {
            const double p0 = __builtin_fma(d.theta1, 0.0, d.theta0);
            const double p1 = __builtin_fma(d.theta1, static_cast<double>(d.len - 1), d.theta0);
            tier = dec_fast_range<T, 1>(p0, p1) ? 1 : (sizeof(T) == 8 && dec_fast_range<T, 2>(p0, p1)) ? 2 : 0;
        }
        L.d[i] = ManyDesc{d.theta0, d.theta1, desc_off(d.packed) - static_cast<int64_t>(sx) * b, sx,
                          static_cast<uint32_t>(d.len), b | (type << 8) | (tier << 12), 0};
        wide |= b > 32 ? 1 : 0;
        return sx;
    });
    if (!ok) return false;
    const bool any_wide = __any(wide) != 0;
    const int32_t cnt = static_cast<int32_t>(e1 - e0);
    int base = 0;  // partitions that start in the rows before
    for (int r0 = 0; r0 < kWaveRows + (SKEW ? 1 : 0); r0 += 4) {
        int idx[4];
        uint32_t w0[4], w1[4], w2[4];
        int64_t pl[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (SKEW && k > 0 && r0 == kWaveRows) break;
            const int32_t x = row_start<SKEW>(r0 + k, a.skew) + lane;
            idx[k] = SKEW ? many_index_at(L.bits, x - lane, row_end<SKEW>(r0 + k, a.skew), lane, base)
                          : many_index(L.bits, r0 + k, lane, base);
            const ManyDesc& d = L.d[idx[k]];
            const bool in = x < cnt && static_cast<uint32_t>(x - d.sx) < d.len;
            if constexpr (OP == OP_PLAIN) {
                pl[k] = a.plain[e0 + (in ? x : 0)];
            } else {
                const int64_t wi = in ? (d.off + static_cast<int64_t>(x) * (d.info & 255)) >> 5 : 0;
                w0[k] = a.words[wi];
                w1[k] = a.words[wi + 1];
                w2[k] = any_wide ? a.words[wi + 2] : 0u;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (SKEW && k > 0 && r0 == kWaveRows) break;
            const int32_t x = row_start<SKEW>(r0 + k, a.skew) + lane;
            const ManyDesc& d = L.d[idx[k]];
            const int32_t i = x - d.sx;
            const int32_t type = (d.info >> 8) & 15;
            O v = O(0);
            if (static_cast<uint32_t>(i) < d.len) {
                uint64_t raw;
                int64_t delta;
                if constexpr (OP == OP_PLAIN) {
                    delta = pl[k];
                    raw = static_cast<uint64_t>(delta);
                } else {
                    const int b = d.info & 255;
                    const uint32_t sh = (static_cast<uint32_t>(d.off) + static_cast<uint32_t>(x) * static_cast<uint32_t>(b)) & 31;
                    const uint32_t f = __builtin_amdgcn_alignbit(w1[k], w0[k], sh);
                    if (any_wide) {  // wave-uniform
                        raw = static_cast<uint64_t>(__builtin_amdgcn_alignbit(w2[k], w1[k], sh)) << 32 | f;
                        delta = sign_extend(raw, b);
                        raw = b >= 64 ? raw : raw & ((1ULL << b) - 1ULL);
                    } else {
                        raw = b == 32 ? f : f & ((1u << b) - 1u);
                        // the builtin returns an unsigned: sign-extend through int32
                        delta = b == 32 ? static_cast<int64_t>(static_cast<int32_t>(f))
                                        : static_cast<int64_t>(static_cast<int32_t>(__builtin_amdgcn_sbfe(
                                              static_cast<int>(f), 0u, static_cast<unsigned>(b))));
                    }
                }
                if constexpr (OP == OP_UNPACK) {
                    v = type == MODEL_DIRECT_COPY ? static_cast<int64_t>(static_cast<T>(raw)) : delta;
                } else {
                    const int tier = d.info >> 12;
                    if (tier == 1) v = apply_delta<T>(dec_pred_fast<T, 1>(d.t0, d.t1, i), delta);
                    else if (sizeof(T) == 8 && tier == 2) v = apply_delta<T>(dec_pred_fast<T, 2>(d.t0, d.t1, i), delta);
                    else if (type == MODEL_DIRECT_COPY) v = static_cast<T>(raw);
                    else
                        v = apply_delta<T>(dec_pred_poly<T>(type, d.t0, d.t1,
                                                            type == MODEL_POLY2 ? a.params[4 * (plo + idx[k]) + 2] : 0.0, i),
                                           delta);
                }
            }
            if (x < cnt && (!SKEW || x < row_end<true>(r0 + k, a.skew))) put(out + x, v);
        }
    }
    return true;
}

// A tile of the partition-spanning path.  VEC: the output is 16-byte aligned; where
// it is not, seg_rows' rows are shifted to its lines.
template <class T, int OP, bool VEC>
__device__ __forceinline__ void wave_segs(const DecArgs& a, int64_t e0, int64_t e1, int64_t plo, int64_t phi,
                                          int lane, ManyLds* L) {
    typedef typename std::conditional<OP == OP_UNPACK, int64_t, T>::type O;
    if (phi - plo >= kSegParts) {
        const int64_t np = phi - plo + 1;
        if (np > kManyParts || !wave_many<T, OP, !VEC>(a, e0, e1, plo, static_cast<int>(np), lane, *L))
            wave_slow<T, OP>(a, e0, e1, plo, lane);
        return;
    }
    O* __restrict__ out = static_cast<O*>(a.out);
    int64_t done = e0;  // everything before is written
    Desc next = a.desc[plo];
    for (int64_t p = plo; p <= phi; ++p) {
        const Desc d = next;
        next = a.desc[p < phi ? p + 1 : p];
        const int64_t ds = d.start, de = ds + d.len;
        const int64_t s = ds > e0 ? ds : e0, t = de < e1 ? de : e1;
        if (s >= t) continue;
        for (int64_t e = done + lane; e < s; e += 64) out[e] = O(0);  // a gap
        seg_decode<T, OP, VEC>(a, d, p, e0, s, t, lane);
        done = t;
    }
    for (int64_t e = done + lane; e < e1; e += 64) out[e] = O(0);
}

// VEC: narrow tiles take the wide-store path (wave_narrow_v), which needs a
// 16-byte aligned output; the host picks the instantiation by the output's
// alignment, so each kernel carries one narrow path only.
// SEGS: partition-spanning tiles take wave_segs.  Its registers (int64: 46 -> 80
// VGPRs packed, 30 -> 60 pre-unpack) move packed and pre-unpacked decodes of columns
// without such tiles by 3 % at most, to either side (without and with, 2^28 int32 215
// and 214 us, int64 491 and 478; 2^27 int64, pre-unpacked, 385 and 391).  Left out of
// batches whose tiles cannot span partitions, of pre-unpacking columns without such
// tiles (2^27 int32: 223 us without, 228 with) and of the half-tile kernel (uint64
// 2^28: 404 us without, 420 with).
template <class T, int OP, bool VEC = true, bool SEGS = false>
__device__ __forceinline__ void wave_tile(const DecArgs& a, int64_t t, int lane, ManyLds* L = nullptr) {
    const int64_t e0 = t * kWaveTile;
    const int64_t e1 = (e0 + kWaveTile < a.n) ? e0 + kWaveTile : a.n;
    const TileInfo x = a.tinfo[t];
    // loaded with the tile's line: spanning tiles need both before anything else
    int64_t plo = 0, phi = 0;
    if constexpr (SEGS) {
        plo = a.tile_part[t];
        phi = a.tile_part[(e1 + kIndexTile - 1) >> kIndexShift];
    }
    const int path = tile_path(x.info);
    if constexpr (OP == OP_PLAIN) {
        if (path != TILE_SLOW) {
            // by halves: with the whole tile in registers the spanning paths run in
            // fewer waves (int64: 79 VGPRs; 5e7 values in partitions of 300 144 -> 151 us)
            for (int h = 0; h < 2; ++h) wave_plain_v<T, 2, !VEC>(a, x, e0, e1, lane, h);
        }
        else if constexpr (SEGS) wave_segs<T, OP, VEC>(a, e0, e1, plo, phi, lane, L);
        else wave_slow<T, OP>(a, e0, e1, a.tile_part[t], lane);
    } else {
        if (path == TILE_NARROW) {
            if constexpr (!VEC) wave_narrow<T>(a, x, e0, e1, lane);
            else if constexpr (OP == OP_UNPACK || sizeof(T) == 8) wave_narrow_v<T, OP, 2>(a, x, e0, e1, lane);
            else if (tile_bits(x.info) <= 16) wave_narrow_v<T, OP, 4>(a, x, e0, e1, lane);
            else wave_narrow_v<T, OP, 2>(a, x, e0, e1, lane);
        }
        else if (path == TILE_WIDE) {
            // shifted rows: two wide fields a lane (1.3e8 int64 values of 41 bits: 312 us, one
            // a lane 330; of 51 bits 330, 350)
            if constexpr (!VEC && SEGS) seg_decode<T, OP, false>(a, a.desc[plo], plo, e0, e0, e1, lane);
            else wave_wide<T, OP>(a, x, e0, e1, lane);
        }
        else if constexpr (SEGS) wave_segs<T, OP, VEC>(a, e0, e1, plo, phi, lane, L);
        else wave_slow<T, OP>(a, e0, e1, a.tile_part[t], lane);
    }
}

// Static grid of one-wave workgroups: workgroup g decodes tile g.  The
// hardware workgroup dispatcher hands tiles to CUs as they free up, and it
// places consecutive workgroups on the XCDs in turn, so consecutive 8-KB
// (64-bit) tiles of the output are written from different XCDs.  Measured on
// the uint64 2^28 column: 0.410 ms against 0.422-0.431 ms with four waves
// (four consecutive tiles) per workgroup; the plain write of 2 GiB in 8-KB
// per-wave runs takes 0.370 ms against 0.397 ms the same way.
template <class T, int OP, bool VEC, bool SEGS, int WPG>
__global__ __launch_bounds__(64 * WPG) void k_decode_wave(DecArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = (WPG == 1) ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t = static_cast<int64_t>(blockIdx.x) * WPG + wave;
    if (t * kWaveTile >= a.n) return;
    if constexpr (SEGS) {
        __shared__ ManyLds L[WPG];
        wave_tile<T, OP, VEC, true>(a, t, lane, &L[wave]);
    } else {
        wave_tile<T, OP, VEC>(a, t, lane);
    }
}

// Pre-unpacked columns of whole-tile partitions: a workgroup of NP waves a tile, a
// part each.  Bound by memory; shorter runs of loads and stores a wave keep both
// going at once (2^27 values, a tile a wave against 4 or 8 parts: int32 283 and 268
// us, int64 384 and 341; the other way round 283 and 367).
template <class T, bool VEC, int NP>
__global__ __launch_bounds__(64 * NP) void k_decode_plain(DecArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t = blockIdx.x;
    const int64_t e0 = t * kWaveTile;
    const int64_t e1 = (e0 + kWaveTile < a.n) ? e0 + kWaveTile : a.n;
    const TileInfo x = a.tinfo[t];
    if (tile_path(x.info) == TILE_SLOW) {  // a gap, or a decode-only polynomial model
        if (wave == static_cast<int>(t % NP)) wave_slow<T, OP_PLAIN>(a, e0, e1, a.tile_part[t], lane);
    } else {
        wave_plain_v<T, NP, !VEC>(a, x, e0, e1, lane, wave);
    }
}

// Half tiles (packed decode into 16-byte aligned outputs; others take whole tiles by
// one wave): one-wave workgroup g decodes half g & 1 of narrow or wide tile g >> 1; a
// tile of any other path is decoded whole by one half's wave, the first's and the
// second's in turn so that every XCD has such waves (all on the first's: 264 instead
// of 166 us, 7e7 uint64 of 36 bits).  (Quarter tiles, one wave per two 128-value rows,
// ran 20-55 % slower on every column measured.)
template <class T>
__global__ __launch_bounds__(64) void k_decode_half(DecArgs a, int64_t ntiles) {
    const int lane = threadIdx.x & 63;
    const int64_t t = static_cast<int64_t>(blockIdx.x) >> 1;
    const int h = static_cast<int>(blockIdx.x & 1);
    if (t >= ntiles) return;
    const TileInfo x = a.tinfo[t];
    const int path = tile_path(x.info);
    const int64_t e0 = t * kWaveTile;
    const int64_t e1 = (e0 + kWaveTile < a.n) ? e0 + kWaveTile : a.n;
    if (path == TILE_WIDE) {
        wave_wide<T, OP_PACKED, 2>(a, x, e0, e1, lane, h);
        return;
    }
    if (path != TILE_NARROW) {  // whole (workgroup g runs on XCD g % 8)
        if (h == static_cast<int>(t >> 2 & 1)) wave_tile<T, OP_PACKED>(a, t, lane);
        return;
    }
    if constexpr (sizeof(T) == 8) wave_narrow_v<T, OP_PACKED, 2, 2>(a, x, e0, e1, lane, h);
    else if (tile_bits(x.info) <= 16) wave_narrow_v<T, OP_PACKED, 4, 2>(a, x, e0, e1, lane, h);
    else wave_narrow_v<T, OP_PACKED, 2, 2>(a, x, e0, e1, lane, h);
}

// Work stealing.  The tiles form 8 contiguous queues, one per XCD (the
// hardware places workgroup b on XCD b % 8).  Every wave the dispatcher
// launches claims the next tile of its XCD's queue with one atomic; when that
// queue is drained it marks it exhausted and steals from the other queues.
// The grid has exactly one wave per tile, so every tile is claimed once.
// Waves are short-lived on purpose: a persistent wave's next loads would
// queue behind its own stores (vmcnt is in-order on gfx9), which halves
// throughput.  The queues are zeroed by a fill kernel before each launch.
constexpr int kStealQueues = 8;
constexpr int kQueueStride = 16;  // ints between queue counters (64 B)

__device__ __forceinline__ int64_t steal_claim(int32_t* q, int qi, int64_t per, int64_t ntiles) {
    for (int tries = 0; tries < kStealQueues; ++tries, qi = (qi + 1) & (kStealQueues - 1)) {
        int32_t* c = q + qi * kQueueStride;
        if (__hip_atomic_load(c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;  // exhausted
        const int64_t base = qi * per;
        const int64_t end = (base + per < ntiles) ? base + per : ntiles;
        int got = 0;
        if ((threadIdx.x & 63) == 0) got = atomicAdd(c, 1);
        got = __builtin_amdgcn_readfirstlane(got);
        if (base + got < end) return base + got;
        if ((threadIdx.x & 63) == 0) __hip_atomic_store(c + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return -1;
}

template <class T, int OP, bool VEC>
__global__ __launch_bounds__(64 * kWavesPerGroup) void k_decode_steal(DecArgs a, int64_t ntiles) {
    const int lane = threadIdx.x & 63;
    const int64_t per = (ntiles + kStealQueues - 1) / kStealQueues;
    const int64_t t = steal_claim(a.sched, static_cast<int>(blockIdx.x & (kStealQueues - 1)), per, ntiles);
    if (t >= 0) wave_tile<T, OP, VEC>(a, t, lane);
}

__global__ void k_zero_queues(int32_t* q) {
    if (threadIdx.x < kStealQueues * kQueueStride) q[threadIdx.x] = 0;
}

// Batched decode: wave (w, k) of workgroup g decodes global tile
// (g*WPG + w)*TPW + k of the batch; the column comes from the tile map and the
// column table (scalar loads), and the element type selects the code path.
// A batch column whose output is not 16-byte aligned: the general per-lane
// path (wave_slow handles every tile kind).  Keeping the one-value-per-lane
// tile bodies out of the batch kernels halves their code (152 KB with them
// for the four element types, more than the instruction cache), and such
// outputs are the exception.
template <class T>
__device__ __forceinline__ void batch_tile_unaligned(const DecArgs& a, int64_t t, int lane) {
    const int64_t e0 = t * kWaveTile;
    const int64_t e1 = (e0 + kWaveTile < a.n) ? e0 + kWaveTile : a.n;
    wave_slow<T, OP_PACKED>(a, e0, e1, a.tile_part[t], lane);
}

template <int WPG, int TPW, bool SEGS>
__global__ __launch_bounds__(64 * WPG) void k_batch_decode(const BatchCol* __restrict__ cols,
                                                           const int32_t* __restrict__ tile_col,
                                                           void* const* __restrict__ outs, int64_t Ttot) {
    const int lane = threadIdx.x & 63;
    const int wave = (WPG == 1) ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ManyLds* L = nullptr;
    if constexpr (SEGS) {
        __shared__ ManyLds s_many[WPG];
        L = &s_many[wave];
    }
    for (int k = 0; k < TPW; ++k) {
        const int64_t g = (static_cast<int64_t>(blockIdx.x) * WPG + wave) * TPW + k;
        if (g >= Ttot) return;
        const int32_t ci = tile_col[g];
        const BatchCol& c = cols[ci];
        DecArgs a;
        a.desc = c.desc;
        a.tile_part = c.tile_part;
        a.words = c.words;
        a.plain = nullptr;
        a.params = c.params;
        a.out = outs[ci];
        a.n = c.n;
        a.P = c.P;
        a.n_index = c.n_index;
        a.tinfo = c.tinfo;
        a.sched = nullptr;
        a.wlimit = c.payload_words;
        a.vec16 = (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
        a.skew = 0;  // outputs that are not aligned take batch_tile_unaligned
        a.pace = a.pace2 = 0;
        const int64_t t = g - c.tile_base;
        if (a.vec16) {
            switch (c.dtype) {
                case GLC_I32: wave_tile<int32_t, OP_PACKED, true, SEGS>(a, t, lane, L); break;
                case GLC_U32: wave_tile<uint32_t, OP_PACKED, true, SEGS>(a, t, lane, L); break;
                case GLC_I64: wave_tile<int64_t, OP_PACKED, true, SEGS>(a, t, lane, L); break;
                default: wave_tile<uint64_t, OP_PACKED, true, SEGS>(a, t, lane, L); break;
            }
        } else {
            switch (c.dtype) {
                case GLC_I32: batch_tile_unaligned<int32_t>(a, t, lane); break;
                case GLC_U32: batch_tile_unaligned<uint32_t>(a, t, lane); break;
                case GLC_I64: batch_tile_unaligned<int64_t>(a, t, lane); break;
                default: batch_tile_unaligned<uint64_t>(a, t, lane); break;
            }
        }
    }
}

// Batched half tiles: one-wave workgroup g decodes half g & 1 of global tile
// g >> 1, the other paths as in k_decode_half.
template <class T, bool SEGS>
__device__ __forceinline__ void batch_half(const DecArgs& a, int64_t t, int h, int lane, ManyLds* L) {
    const TileInfo x = a.tinfo[t];
    const int path = tile_path(x.info);
    const int64_t e0 = t * kWaveTile;
    const int64_t e1 = (e0 + kWaveTile < a.n) ? e0 + kWaveTile : a.n;
    if (path == TILE_WIDE) {
        wave_wide<T, OP_PACKED, 2>(a, x, e0, e1, lane, h);
        return;
    }
    if (path != TILE_NARROW || !a.vec16) {
        if (h == static_cast<int>(t >> 2 & 1)) {
            if (a.vec16) wave_tile<T, OP_PACKED, true, SEGS>(a, t, lane, L);
            else batch_tile_unaligned<T>(a, t, lane);
        }
        return;
    }
    if constexpr (sizeof(T) == 8) wave_narrow_v<T, OP_PACKED, 2, 2>(a, x, e0, e1, lane, h);
    else if (tile_bits(x.info) <= 16) wave_narrow_v<T, OP_PACKED, 4, 2>(a, x, e0, e1, lane, h);
    else wave_narrow_v<T, OP_PACKED, 2, 2>(a, x, e0, e1, lane, h);
}

template <bool SEGS>
__global__ __launch_bounds__(64) void k_batch_decode_half(const BatchCol* __restrict__ cols,
                                                          const int32_t* __restrict__ tile_col,
                                                          void* const* __restrict__ outs, int64_t Ttot) {
    const int lane = threadIdx.x & 63;
    ManyLds* L = nullptr;
    if constexpr (SEGS) {
        __shared__ ManyLds s_many;
        L = &s_many;
    }
    const int64_t g = static_cast<int64_t>(blockIdx.x) >> 1;
    const int h = static_cast<int>(blockIdx.x & 1);
    if (g >= Ttot) return;
    const int32_t ci = tile_col[g];
    const BatchCol& c = cols[ci];
    DecArgs a;
    a.desc = c.desc;
    a.tile_part = c.tile_part;
    a.words = c.words;
    a.plain = nullptr;
    a.params = c.params;
    a.out = outs[ci];
    a.n = c.n;
    a.P = c.P;
    a.n_index = c.n_index;
    a.tinfo = c.tinfo;
    a.sched = nullptr;
    a.wlimit = c.payload_words;
    a.vec16 = (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
    a.skew = 0;
    a.pace = a.pace2 = 0;
    const int64_t t = g - c.tile_base;
    switch (c.dtype) {
        case GLC_I32: batch_half<int32_t, SEGS>(a, t, h, lane, L); break;
        case GLC_U32: batch_half<uint32_t, SEGS>(a, t, h, lane, L); break;
        case GLC_I64: batch_half<int64_t, SEGS>(a, t, h, lane, L); break;
        default: batch_half<uint64_t, SEGS>(a, t, h, lane, L); break;
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

DecArgs make_args(const glc_column* c, void* out) {
    DecArgs a;
    a.desc = c->d_desc;
    a.tile_part = c->d_tile_part;
    // The tile paths load words whatever the width.  A released payload of no bits
    // (glc_preunpack with free_packed; launch_decode_full refuses others): every
    // load is within 128 + 64 words of its first one, and what it brings is masked
    // to 0 bits, so any 1 KiB of the column's own arena does.
    static_assert(kSchedBytes >= kPayloadPadWords * 4, "the queues' part alone covers the loads");
    a.words = c->d_words ? c->d_words : static_cast<const uint32_t*>(c->meta_arena);
    a.plain = c->d_plain;
    a.params = c->d_params;
    a.out = out;
    a.n = c->n;
    a.P = c->P;
    a.n_index = c->n_index;
    a.tinfo = c->d_tinfo;
    a.wlimit = c->payload_words;
    a.sched = c->d_sched;
    a.vec16 = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    a.skew = static_cast<int32_t>((reinterpret_cast<uintptr_t>(out) & 127) / c->elem_size);
    a.spans = c->spans;
    a.wide = c->max_bits > 32;
    a.pace = a.pace2 = c->dec_pace;
    return a;
}

template <class T, int OP, bool VEC, bool SEGS>
void launch_static(const DecArgs& a, int dsched, int64_t nwt, hipStream_t s) {
    if (dsched == GLC_DECODE_HALF_TILE_W1 && OP == OP_PACKED && VEC)
        hipLaunchKernelGGL(k_decode_half<T>, dim3(static_cast<unsigned>(2 * nwt)), dim3(64), 0, s, a, nwt);
    else if (dsched != GLC_DECODE_TILE_W4)
        hipLaunchKernelGGL((k_decode_wave<T, OP, VEC, SEGS, 1>), dim3(static_cast<unsigned>(nwt)), dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL((k_decode_wave<T, OP, VEC, SEGS, 4>), dim3(static_cast<unsigned>((nwt + 3) / 4)), dim3(256),
                           0, s, a);
}

template <class T, int OP> int run(const DecArgs& a, int sched, hipStream_t s, int dsched = GLC_DECODE_TILE_W4) {
    const int64_t nwt = (a.n + kWaveTile - 1) / kWaveTile;
    switch (sched) {
        case 0:
            if constexpr (OP == OP_UNPACK) {  // into its own block, aligned; wave_tile's note
                if (a.spans) launch_static<T, OP, true, true>(a, dsched, nwt, s);
                else launch_static<T, OP, true, false>(a, dsched, nwt, s);
            } else if (OP == OP_PLAIN && !a.spans) {
                constexpr int kParts = sizeof(T) == 8 ? 8 : 4;
                const dim3 g(static_cast<unsigned>(nwt));
                if (a.vec16) hipLaunchKernelGGL((k_decode_plain<T, true, kParts>), g, dim3(64 * kParts), 0, s, a);
                else hipLaunchKernelGGL((k_decode_plain<T, false, kParts>), g, dim3(64 * kParts), 0, s, a);
            } else if (a.vec16) {
                launch_static<T, OP, true, true>(a, dsched, nwt, s);
            } else if (OP == OP_PLAIN || a.spans || a.wide) {
                launch_static<T, OP, false, true>(a, dsched, nwt, s);
            } else {
                launch_static<T, OP, false, OP == OP_PLAIN>(a, dsched, nwt, s);
            }
            break;
        case 1: {
            hipLaunchKernelGGL(k_zero_queues, dim3(1), dim3(kStealQueues * kQueueStride), 0, s, a.sched);
            if (a.vec16)
                hipLaunchKernelGGL((k_decode_steal<T, OP, true>),
                                   dim3(static_cast<unsigned>((nwt + kWavesPerGroup - 1) / kWavesPerGroup)),
                                   dim3(64 * kWavesPerGroup), 0, s, a, nwt);
            else
                hipLaunchKernelGGL((k_decode_steal<T, OP, false>),
                                   dim3(static_cast<unsigned>((nwt + kWavesPerGroup - 1) / kWavesPerGroup)),
                                   dim3(64 * kWavesPerGroup), 0, s, a, nwt);
            break;
        }
        default: return fail(GLC_ERR_INVALID_ARG, "bad schedule");
    }
    GLC_HIP(hipGetLastError());
    return GLC_OK;
}

}  // namespace

int launch_decode_full(const glc_column* c, void* d_out, int mode, hipStream_t s) {
    if (c->n == 0) return GLC_OK;
    bool plain;
    int sched;
    switch (mode) {
        case GLC_FULL_AUTO: plain = c->d_plain != nullptr; sched = 0; break;
        case GLC_FULL_BITPACKED: plain = false; sched = 0; break;
        case GLC_FULL_PREUNPACKED: plain = true; sched = 0; break;
        case GLC_FULL_V2: plain = c->d_plain != nullptr; sched = 0; break;
        // Work stealing: tiles are claimed by CUs as they free up through the
        // hardware workgroup dispatcher (one short-lived wave per 1024-value
        // tile).  Explicit claims through device-scope atomics (kModeWaveSteal)
        // serialize at ~14 ns per claim: 3.8 ms against 0.43-0.48 ms for the
        // 2^18 tiles of a 2^28-value column.
        case GLC_FULL_WORKSTEAL: plain = c->d_plain != nullptr; sched = 0; break;
        case GLC_FULL_WORKSTEAL_ADV: plain = c->d_plain != nullptr; sched = 0; break;
        case GLC_FULL_COOP_EXACT: plain = true; sched = 0; break;
        // the explicit work-stealing comparator of WorkStealingDecompressionKernels.cuh:332-521:
        // wave tiles claimed from per-XCD atomic queues
        case kModeWaveSteal: plain = c->d_plain != nullptr; sched = 1; break;
        default: return fail(GLC_ERR_INVALID_ARG, "bad full-decompress mode");
    }
    if (plain && !c->d_plain)
        return fail(GLC_ERR_UNSUPPORTED, "no pre-unpacked deltas (call glc_preunpack or deserialize with preunpack)");
    if (!plain && !c->d_words && c->total_bits > 0)
        return fail(GLC_ERR_UNSUPPORTED, "bit-packed payload was released by glc_preunpack(free_packed=1)");
    if (c->P == 0) return fail(GLC_ERR_STATE, "column has values but no partitions");
    DecArgs a = make_args(c, d_out);
    // No schedule set: 64-bit columns of whole-tile partitions take half tiles
    // (2^28 values 399-560 us against 431-631 with four tiles a workgroup, by width;
    // within 3 % below 2^27).  Long ones of wide fields whose predictions are beyond
    // 2^50 (timestamps) also space their stores out: 2^28 values of 17 / 19 / 21 / 24 / 29
    // bits take 411 / 422 / 463 / 478 / 512 us without, 454 / 452 / 449 / 446 / 497 with;
    // 2^26 of 20 bits 106 and 109.  32-bit columns are faster in whole tiles (2^28 239-278
    // against 254-291), and the half-tile kernel has no fast path for
    // partition-spanning tiles and none for outputs that are not 16-byte aligned.
    // Those decode in one-wave workgroups (1.3e8 int64 values of 41 bits, S = 1000: 321
    // us in fours, 316 so; S = 3000: 351, 331, and of 13 bits 244, 236; int32 of 25 bits
    // 187, 178).
    int dsched = c->dec_sched;
    if (c->dec_auto && !a.vec16) {
        dsched = GLC_DECODE_TILE_W1;
    } else if (c->dec_auto && c->elem_size == 8 && !c->spans) {
        dsched = GLC_DECODE_HALF_TILE_W1;
        if (c->n >= (int64_t(1) << 27) && c->total_bits >= 21 * c->n) a.pace2 = 16;
    }
    return dispatch_dtype(c->dtype, [&](auto t) {
        using T = decltype(t);
        return plain ? run<T, OP_PLAIN>(a, sched, s, c->dec_sched) : run<T, OP_PACKED>(a, sched, s, dsched);
    });
}

int glc_autotune_decode(glc_column* c, void* d_out, int32_t reps, hipStream_t s, int32_t* best_out, float* ms_out) {
    if (c->n == 0 || c->P == 0 || (!c->d_words && c->total_bits > 0)) {
        if (best_out) *best_out = c->dec_sched;
        if (ms_out) *ms_out = 0.0f;
        return GLC_OK;
    }
    // every schedule with every pace
    constexpr int kS = 3, kPaces = 5, kC = kS * kPaces;
    const int sched_of[kS] = {GLC_DECODE_TILE_W1, GLC_DECODE_TILE_W4, GLC_DECODE_HALF_TILE_W1};
    const int pace_of[kPaces] = {0, 4, 8, 16, 24};
    const int saved = c->dec_sched, saved_pace = c->dec_pace;
    const bool saved_auto = c->dec_auto;
    c->dec_auto = false;
    std::vector<hipEvent_t> ev(static_cast<size_t>(2 * kC * reps), nullptr);
    int rc = GLC_OK;
    for (auto& e : ev)
        if (hipEventCreate(&e) != hipSuccess) {
            e = nullptr;
            rc = fail(GLC_ERR_HIP, "hipEventCreate failed");
            break;
        }
    auto set = [&](int k) {
        c->dec_sched = sched_of[k / kPaces];
        c->dec_pace = pace_of[k % kPaces];
    };
    // one warm-up launch per combination, then `reps` rounds over them
    // (round-robin, so clock and cache drift falls on every one alike)
    for (int k = 0; k < kC && !rc; ++k) {
        set(k);
        rc = launch_decode_full(c, d_out, GLC_FULL_BITPACKED, s);
    }
    for (int r = 0; r < reps && !rc; ++r)
        for (int k = 0; k < kC && !rc; ++k) {
            set(k);
            const size_t i = static_cast<size_t>(2 * (r * kC + k));
            if (hipEventRecord(ev[i], s) != hipSuccess) rc = fail(GLC_ERR_HIP, "hipEventRecord failed");
            if (!rc) rc = launch_decode_full(c, d_out, GLC_FULL_BITPACKED, s);
            if (!rc && hipEventRecord(ev[i + 1], s) != hipSuccess) rc = fail(GLC_ERR_HIP, "hipEventRecord failed");
        }
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = fail(GLC_ERR_HIP, "hipStreamSynchronize failed");
    int best = -1;
    float best_ms = 0.0f;
    if (!rc) {
        for (int k = 0; k < kC; ++k) {  // median launch time of each combination
            std::vector<float> t(static_cast<size_t>(reps));
            for (int r = 0; r < reps; ++r) {
                const size_t i = static_cast<size_t>(2 * (r * kC + k));
                (void)hipEventElapsedTime(&t[static_cast<size_t>(r)], ev[i], ev[i + 1]);
            }
            std::sort(t.begin(), t.end());
            const float med = t[t.size() / 2];
            if (best < 0 || med < best_ms) {
                best_ms = med;
                best = k;
            }
        }
    }
    for (auto& e : ev)
        if (e) (void)hipEventDestroy(e);
    if (rc || best < 0) {
        c->dec_sched = saved;
        c->dec_pace = saved_pace;
        c->dec_auto = saved_auto;
        return rc;
    }
    set(best);
    if (best_out) *best_out = c->dec_sched;
    if (ms_out) *ms_out = best_ms;
    return rc;
}

int launch_batch_decode(const BatchPlan& b, int wpg, int tpw, hipStream_t s) {
    if (b.Ttot == 0) return GLC_OK;
    auto grid = [&](int w, int t) {
        return dim3(static_cast<unsigned>((b.Ttot + static_cast<int64_t>(w) * t - 1) / (static_cast<int64_t>(w) * t)));
    };
    // partitions that are no multiple of a tile leave partition-spanning tiles
    // all over: the instantiations with the spanning paths
    const bool segs = b.S % kIndexTile != 0;
#define GLC_BATCH_CASE(W, TP)                                                                                     \
    if (wpg == W && tpw == TP) {                                                                                  \
        if (segs)                                                                                                 \
            hipLaunchKernelGGL((k_batch_decode<W, TP, true>), grid(W, TP), dim3(64 * W), 0, s, b.cols, b.tile_col, \
                               b.outs, b.Ttot);                                                                   \
        else                                                                                                      \
            hipLaunchKernelGGL((k_batch_decode<W, TP, false>), grid(W, TP), dim3(64 * W), 0, s, b.cols,           \
                               b.tile_col, b.outs, b.Ttot);                                                       \
        GLC_HIP(hipGetLastError());                                                                               \
        return GLC_OK;                                                                                            \
    }
    GLC_BATCH_CASE(4, 1)
    GLC_BATCH_CASE(2, 1)
    GLC_BATCH_CASE(8, 1)
    GLC_BATCH_CASE(1, 1)
    GLC_BATCH_CASE(4, 2)
    GLC_BATCH_CASE(2, 4)
#undef GLC_BATCH_CASE
    if (wpg == 1 && tpw == 0) {
        const dim3 g(static_cast<unsigned>(2 * b.Ttot));
        if (segs) hipLaunchKernelGGL(k_batch_decode_half<true>, g, dim3(64), 0, s, b.cols, b.tile_col, b.outs, b.Ttot);
        else hipLaunchKernelGGL(k_batch_decode_half<false>, g, dim3(64), 0, s, b.cols, b.tile_col, b.outs, b.Ttot);
        GLC_HIP(hipGetLastError());
        return GLC_OK;
    }
    return fail(GLC_ERR_INVALID_ARG, "unsupported batch schedule");
}

int launch_preunpack(glc_column* c, int64_t* d_plain, hipStream_t s) {
    if (c->n == 0) return GLC_OK;
    DecArgs a = make_args(c, d_plain);
    return dispatch_dtype(c->dtype, [&](auto t) {
        using T = decltype(t);
        return run<T, OP_UNPACK>(a, 0, s);
    });
}

}  // namespace glc
