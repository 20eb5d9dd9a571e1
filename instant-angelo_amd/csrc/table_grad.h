// Deterministic table-gradient reduction: (row, value) pairs emitted by a
// backward kernel -> one write per row of the table gradient, rows without a
// pair written 0, the same bits on every run.
//
// Paged form (two features a row, at most 2^21 rows a level: every grid of
// the workloads).  The emitters write one stream of pairs per level.  A
// stream is cut into pages of kPage pairs; each page is partitioned in place
// (in LDS) by its pairs' bucket of 2^13 rows, with a table of where each
// bucket's run starts, and one block per bucket then gathers its runs from
// the level's pages and adds them up in LDS.  The additions are exact (see
// k_page_reduce), so their order does not matter.
//
// Sorted form (other feature counts, larger levels): stable radix sort of the
// pairs by row, then a fixed-order segmented reduce.  Two-feature tables sort
// only the key bits above `begin_bit`: the pairs of each bucket of
// 2^begin_bit rows are then contiguous and in emission order, and one wave
// per bucket finishes the job with an in-wave stable split sort and a
// segmented scan into per-row accumulators in LDS.
//
// The emitters write pairs into carve.keys[0] / carve.vals[0] (keys: table
// rows).
#pragma once
#include <hip/hip_fp16.h>
#include "am_common.h"

namespace am {

template <int F>
struct Vals {
    float v[F];
};

// Pair values stored in fp16 (the mixed-precision form: loss-scaled
// gradients, summed in fp32 by the segmented reduce).
template <int F>
struct ValsH {
    __half v[F];
};

constexpr int kSegChunk = 17;  // items reduced sequentially per thread (odd: LDS banks)

struct TableReduceWs {
    uint32_t* keys[2];
    void* vals[2];
    void* sort_tmp;
    size_t sort_bytes;
    float* lead;
    float* tail;
    uint8_t* lead_full;
    uint8_t* tail_open;
    int64_t* bucket_start;  // [n_buckets + 1] (bucketed form)
    uint64_t* units;        // [n_buckets + 1] packed work-unit counts
    uint64_t* unit_off;     // [n_buckets + 1] their exclusive scan
    float* partial;         // partial sums of multi-unit buckets
    void* scan_tmp;
    size_t scan_bytes;
    int64_t n_buckets;      // 0: full sort + chunked segmented reduce
    int64_t m;
    int begin_bit;          // key bits sorted: [begin_bit, end_bit)
    int end_bit;
    bool half_vals;  // values are ValsH<F> instead of Vals<F>
    bool paged;      // paged form: the fields below
    uint16_t* run_start;    // [pages][kRunStride] first pair of each bucket's run
    double2* partial2;      // [slots][8192 rows] sums of sliced buckets
    struct PagePlan* plan;
    int64_t* level_start;   // [levels + 1] first pair of each level's stream
};

// Rows of the levels: level l owns [offset[l], offset[l + 1]).
struct TableLevels {
    int32_t L;
    uint32_t offset[AM_MAX_LEVELS + 1];
};
TableLevels table_levels(const am_grid_desc* g);

// What the paged kernels read of the streams (made on the device from
// level_start, so that no host read is needed).
struct PagePlan {
    int64_t level_start[AM_MAX_LEVELS + 1];
    int32_t page_base[AM_MAX_LEVELS + 1];   // first page of each level
    int32_t unit_base[AM_MAX_LEVELS + 1];   // first work unit of each level (finest level first)
    int32_t slices[AM_MAX_LEVELS];          // slices of each of the level's buckets
    int32_t slot_base[AM_MAX_LEVELS];       // first partial slot of a sliced level
    int32_t row_base[AM_MAX_LEVELS + 1];    // first combined row of a sliced level
};

// Bucket bits of the bucketed form: the low key bits left unsorted (at most
// 9, so a wave's accumulators span at most 512 rows).
int table_bucket_bits(int end_bit);

// Number of key bits: smallest b with 2^b > n_entries (so the sentinel
// (2^b - 1) is >= n_entries and never a valid row).
int table_key_bits(uint32_t n_entries);
static inline uint32_t table_sentinel(int end_bit) { return (uint32_t)((1ull << end_bit) - 1ull); }

// Carves the reduction workspace for m pairs out of `c`.  Returns the sort's
// temp byte count through TableReduceWs (0 when c has no base pointer: size
// query; the sort size query needs a device).
int table_reduce_carve(WsCarver& c, const am_grid_desc* g, int64_t m, TableReduceWs* out,
                       bool half_vals = false);

// Writes v to p[0..n) on `stream` (a fill kernel, safe under graph capture).
int fill_f32(float* p, int64_t n, float v, hipStream_t stream);

// Reduces the pairs; dtable [n_entries, F] fully overwritten.  Paged form:
// w.level_start holds the level streams' bounds (at most w.m pairs); sorted
// form: exactly w.m pairs (sentinel keys allowed).
int table_reduce_run(TableReduceWs& w, const am_grid_desc* g, float* dtable, hipStream_t stream);

}  // namespace am
