// Table-gradient pairs of the fused SDF field's backward (pairs.hip).
#pragma once
#include "geo_args.h"

namespace am {

// What the passes need before the pair arrays are carved.
struct PairHead {
    bool paged;            // pages (page_dev.h), or arrays for the sorted form
    int64_t* status;       // [0] pages (paged) or pairs, [1] consistency flag, [2] pairs
    // paged
    float* centers;        // [6][samples, whole blocks] cluster centres
    uint32_t* steps;       // [units][kPairSteps] pairs of each emission step
    uint64_t* unit_pages;  // [units + 1] pages << 40 | pairs
    uint64_t* unit_scan;   // its exclusive scan
    int64_t units;         // active levels x sample blocks
    // sorted
    int64_t* counts;       // [levels][tiles]
    int64_t* offsets;
    int64_t entries;
    void* scan_tmp;
    size_t scan_bytes;
};

void pairs_carve(WsCarver& c, const GeoArgs& a, const am_grid_desc* g, int64_t n, PairHead* h);
// Count pass and scan; h.status[0] = capacity the emission needs (pages, or
// pairs), h.status[2] = pairs.
int pairs_count(const GeoArgs& a, int LJ, const float* pts, const float* randn, int64_t n,
                const float* fdv, PairHead& h, hipStream_t s);
// The most status[0] can be for n samples.
int64_t pairs_bound(const GeoArgs& a, const PairHead& h, int LJ, int64_t n);
// Emission and reduction into dtable.
int pairs_reduce(const GeoArgs& a, int LJ, const am_grid_desc* g, const float* pts,
                 const float* randn, int64_t n, const float* fdv, const float* genc, PairHead& h,
                 TablePages& tp, TableReduceWs& tw, bool bounded, float* dtable, hipStream_t s);
// The merged pairs added into the zeroed dtable with float atomics.
int pairs_atomic(const GeoArgs& a, int LJ, const float* pts, const float* randn, int64_t n,
                 const float* fdv, const float* genc, float* dtable, hipStream_t s);

}  // namespace am
