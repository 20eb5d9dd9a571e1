// Pages of table-gradient pairs: what the emitting kernels (pairs.hip,
// hashgrid.hip) and the reduction (table_grad.hip) share.
#pragma once
#include "table_grad.h"

namespace am {

// A page: up to kPage pairs of one level, partitioned by their bucket of
// kRows rows.  Its key words hold the row within the bucket (bits 0-12) and
// the two values' exponents (13-20, 21-28); run_start[page][b] is the first
// pair of bucket b's run.
constexpr int kPage = 12288;         // with fp32 values a page fills a CU's LDS
constexpr int kPageThreads = 1024;
constexpr int kRowBits = 13;         // rows a bucket: its sums fill the reduce's LDS
constexpr int kRows = 1 << kRowBits;
constexpr int kMaxDigits = 256;      // buckets a level: 2^21 rows
constexpr int kRunStride = kMaxDigits + 2;

__device__ __forceinline__ float2 pair_value(uint2 v) {
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}
__device__ __forceinline__ float2 pair_value(uint32_t v) {
    return __half22float2(__builtin_bit_cast(__half2, v));
}
// Inclusive sum over the wave's lanes.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if ((int)(threadIdx.x & 63) >= d) v += o;
    }
    return v;
}

// The page under construction: pairs in any order (keys: rows within the
// level).  hist is zero between flushes.
// Values are kept by word (fp32: the first features, then the second ones;
// fp16: the pairs).
template <class VT>
struct PageLds {
    uint32_t words[sizeof(VT) / 4][kPage];
    uint32_t keys[kPage];
    uint32_t hist[kMaxDigits + 4];
    uint32_t cursor;   // pairs put so far
};

__device__ __forceinline__ void page_put(PageLds<uint2>& s, int at, uint32_t row, float a, float b) {
    s.keys[at] = row;
    s.words[0][at] = __float_as_uint(a);
    s.words[1][at] = __float_as_uint(b);
}
__device__ __forceinline__ void page_put(PageLds<uint32_t>& s, int at, uint32_t row, float a,
                                         float b) {
    s.keys[at] = row;
    s.words[0][at] =
        __builtin_bit_cast(uint32_t, __halves2half2(__float2half_rn(a), __float2half_rn(b)));
}
__device__ __forceinline__ uint2 page_value(const PageLds<uint2>& s, int i) {
    return make_uint2(s.words[0][i], s.words[1][i]);
}
__device__ __forceinline__ uint32_t page_value(const PageLds<uint32_t>& s, int i) {
    return s.words[0][i];
}

// Partitions the LDS page's n pairs by bucket and writes them to page `page`.
// The runs hold their pairs in any order (the reduce's sums do not depend on
// it), so each pair's place comes from one LDS counter.  spread (levels of
// few buckets, whose runs are long and full of repeated rows): pairs that
// arrive together, neighbouring samples often of one row, are set a wave's
// load apart, so that the reduce's LDS additions seldom meet in one row (60 M
// pairs in runs of 16 equal rows: reduce 0.80 -> 0.34 ms).  The second
// features move after the others, to hold few registers beside the caller's.
// Bound by LDS operations.  Called by all kPageThreads threads; leaves the
// page empty.  mismatch (null: n is what was put): set to 1 when the pairs put
// (cursor) are not the n counted; only pairs that were both put and counted are
// written then.
template <class VT>
__device__ __forceinline__ void page_flush(PageLds<VT>& s, int n, int64_t* __restrict__ mismatch,
                                           bool spread, int64_t page,
                                           uint32_t* __restrict__ keys, VT* __restrict__ vals,
                                           uint16_t* __restrict__ run_start) {
    constexpr int kItems = kPage / kPageThreads;
    int tid = (int)threadIdx.x;
    asm volatile("" : "+v"(tid));   // keeps its addresses out of the caller's loop registers
    uint32_t key[kItems], at[kItems], first[kItems];   // first: words[0]
    __syncthreads();
    if (mismatch) {
        const int put = __builtin_amdgcn_readfirstlane((int)s.cursor);
        if (put != n && tid == 0) *mismatch = 1;
        n = put < n ? put : n;
    }
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int i = tid + kPageThreads * k;
        if (i < n) {
            key[k] = s.keys[i];
            at[k] = atomicAdd(&s.hist[(key[k] >> kRowBits) & (uint32_t)(kMaxDigits - 1)], 1u);
        }
        if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    if (tid < 64) {   // four counters a lane
        uint32_t c[4];
        uint32_t sum = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            c[q] = sum;
            sum += s.hist[4 * tid + q];
        }
        const uint32_t before = wave_scan(sum) - sum;
        uint16_t* rs = run_start + page * kRunStride;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            s.hist[4 * tid + q] = before + c[q];
            rs[4 * tid + q] = (uint16_t)(before + c[q]);
        }
        if (tid == 63) {
            s.hist[kMaxDigits] = (uint32_t)n;
            rs[kMaxDigits] = (uint16_t)n;
            s.cursor = 0u;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (tid + kPageThreads * k < n) {
            const uint32_t d = (key[k] >> kRowBits) & (uint32_t)(kMaxDigits - 1);
            const uint32_t h0 = s.hist[d];
            uint32_t r = at[k];
            if (spread) {
                const uint32_t q = (s.hist[d + 1] - h0) >> 6;
                if (q > 1u && r < q << 6) {   // r = a q + b -> 64 b + a
                    const uint32_t a =
                        (uint32_t)(((float)r + 0.5f) * __builtin_amdgcn_rcpf((float)q));
                    r = (r - a * q) * 64u + a;
                }
            }
            r += h0;
            at[k] = r;
            const int i = tid + kPageThreads * k;
            const float2 f = pair_value(page_value(s, i));
            first[k] = s.words[0][i];
            key[k] = (key[k] & (uint32_t)(kRows - 1)) |
                     (__float_as_uint(f.x) >> 23 & 255u) << kRowBits |
                     (__float_as_uint(f.y) >> 23 & 255u) << (kRowBits + 8);
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (tid + kPageThreads * k < n) {
            s.keys[at[k]] = key[k];
            s.words[0][at[k]] = first[k];
        }
    if constexpr (sizeof(VT) == 8) {
#pragma unroll
        for (int k = 0; k < kItems; ++k)
            if (tid + kPageThreads * k < n) first[k] = s.words[1][tid + kPageThreads * k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kItems; ++k)
            if (tid + kPageThreads * k < n) s.words[1][at[k]] = first[k];
    }
    __syncthreads();
    keys += page * kPage;
    vals += page * kPage;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int i = tid + kPageThreads * k;
        if (i < n) {
            keys[i] = s.keys[i];
            vals[i] = page_value(s, i);
        }
        if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if (tid <= kMaxDigits) s.hist[tid] = 0u;
    __syncthreads();
}

// A page without pairs (one that the emission did not reach).
__device__ __forceinline__ void page_empty(int64_t page, uint16_t* __restrict__ run_start) {
    if ((int)threadIdx.x <= kMaxDigits) run_start[page * kRunStride + threadIdx.x] = 0;
}

// Levels of at most this many buckets spread their runs.
constexpr int kSpreadDigits = 96;

}  // namespace am
