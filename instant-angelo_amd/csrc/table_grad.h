// Deterministic table-gradient reduction: (row, value) pairs emitted by a
// backward kernel -> one write per row of the table gradient, rows without a
// pair written 0, the same bits on every run.
//
// Paged form (two features a row, at most 2^21 rows a level, the levels one
// after another: every grid of the workloads).  The emitting kernels collect
// the pairs of one level in LDS, a page at a time, and write each page
// partitioned by its pairs' bucket of 2^13 rows, with a table of where each
// bucket's run starts; one block per bucket then gathers its runs from the
// level's pages and adds them up in LDS.  The additions are exact (see
// k_page_reduce), so their order does not matter.  Every pair is written once
// and its value read once.
//
// Sorted form (other feature counts, larger levels, other layouts): stable
// radix sort of the pairs by row, then a fixed-order segmented reduce.
// Two-feature tables sort only the key bits above `begin_bit`: the pairs of
// each bucket of 2^begin_bit rows are then contiguous and in emission order,
// and one wave per bucket finishes the job with an in-wave stable split sort
// and a segmented scan into per-row accumulators in LDS.
//
// There the emitters write pairs into keys[0] / vals[0].  Keys equal to the
// sentinel mark empty slots; they sort last and are skipped.
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
};

// Rows of the levels: level l owns [offset[l], offset[l + 1]).  Its buckets:
// from bucket[l] on, n_buckets in all.
struct TableLevels {
    int32_t L;
    uint32_t offset[AM_MAX_LEVELS + 1];
    int32_t bucket[AM_MAX_LEVELS];
    int32_t n_buckets;
};
TableLevels table_levels(const am_grid_desc* g);

// What the reduction does (made on the device from the pages' run tables, so
// that no host read is needed).
struct PagePlan {
    int32_t n_units, n_merges;
};
// A bucket's pairs, or (slices > 1) those of every slices-th page, the slice-th
// on.
struct __attribute__((aligned(32))) PageUnit {
    int64_t page;            // the first of them
    int32_t runs, slices;    // pages, and from one to the next
    int32_t bucket;          // within its level
    uint32_t row, rows;      // the bucket's first row, and how many
    int32_t slot;            // partial slot (slices > 1)
};

// Where the pages of each level begin, on the device: the level's `units`
// emitting blocks' exclusive scan (high 24 bits: pages), unit = level * units +
// block, levels from `active` on empty; or (scan == nullptr) `per_level` pages
// for each of the `active` levels.  Never past the arrays' `capacity`.
struct PageSource {
    const uint64_t* scan;
    int64_t units;
    int32_t active;
    int64_t per_level;
    int64_t capacity;
};

struct TablePages {
    int64_t pages;       // the arrays' capacity
    uint32_t* keys;      // [pages][kPage]
    void* vals;          // the same: float2, or half2 (half_vals)
    uint16_t* run_start; // [pages][kRunStride]
    double2* partial;    // [slots][8192 rows] sums of sliced buckets
    int32_t chunks;      // parts of a level's pages counted by a block each (0: few pages)
    uint32_t* pairs;     // [chunks][n_buckets] pairs of the buckets
    PagePlan* plan;
    PageUnit* units;     // [max_units]
    PageUnit* merges;    // [n_buckets] those of several slices, or of no pair (slices 0)
    int64_t max_units;
    bool half_vals;
};

// Whether the paged form takes the grid.
bool table_paged(const am_grid_desc* g);
void table_pages_carve(WsCarver& c, const am_grid_desc* g, int64_t pages, bool half_vals,
                       TablePages* out);
// Reduces the pages (of PageSource); dtable [n_entries, 2] fully overwritten.
int table_pages_run(TablePages& w, const am_grid_desc* g, const uint64_t* scan, int64_t units,
                    int active, int64_t per_level, float* dtable, hipStream_t s);

// ---- sorted form ----
// Bucket bits of the bucketed form: the low key bits left unsorted (at most
// 9, so a wave's accumulators span at most 512 rows).
int table_bucket_bits(int end_bit);

// Number of key bits: smallest b with 2^b > n_entries (so the sentinel
// (2^b - 1) is >= n_entries and never a valid row).
int table_key_bits(uint32_t n_entries);
static inline uint32_t table_sentinel(int end_bit) { return (uint32_t)((1ull << end_bit) - 1ull); }

// Carves the sorted form's workspace for m pairs out of `c`.  Returns the
// sort's temp byte count through TableReduceWs (0 when c has no base pointer:
// size query; the sort size query needs a device).
int table_reduce_carve(WsCarver& c, const am_grid_desc* g, int64_t m, TableReduceWs* out,
                       bool half_vals = false);

// Writes v to p[0..n) on `stream` (a fill kernel, safe under graph capture).
int fill_f32(float* p, int64_t n, float v, hipStream_t stream);

// Runs sort + segmented reduce; dtable [n_entries, F] fully overwritten.
int table_reduce_run(TableReduceWs& w, const am_grid_desc* g, float* dtable, hipStream_t stream);

}  // namespace am
