// Table-gradient pairs of the fused SDF field's backward: turns each sample's
// encode gradients into (row, value) pairs, merged where its evaluations
// share cells.
//   1. Per sample and level, the evaluations of a cluster (base + 6 FD, or the
//      6 curvature points) are merged into the cell B of the cluster centre
//      with a star stencil: an evaluation in B adds its 8 corners, one in a
//      face neighbour of B adds the 4 corners of the shared face and emits
//      its 4 far corners, any other emits its 8 corners.
//   2. B's corner sums are merged with equal-B lanes of the same 16 lanes
//      (neighbouring samples of a ray) by a segmented reduction in a fixed
//      shuffle tree.
//   3. A count pass makes the same decisions from positions alone and sizes
//      the pages (paged form) or the arrays (sorted form).
#include "pairs.h"
#include "page_dev.h"
#include "field_common.h"
#include <rocprim/device/device_scan.hpp>

namespace am {

// Lane p + D (p - 1) of the lane's 16-lane row (a DPP row shift: no LDS
// traffic); lanes whose source lies outside the row get 0 and must not use it.
template <int D>
__device__ __forceinline__ uint32_t row_down(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + D, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t row_up1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
}

// One step of the suffix segmented sum over a 16-lane row: a lane that is
// not the end of its segment adds the accumulators of lane p + D (and takes
// over its end flag) when that lane is in the row.
template <int D>
__device__ __forceinline__ void merge_step(int p, float acc[16], bool& end) {
    float o[16];
#pragma unroll
    for (int c = 0; c < 16; ++c)
        o[c] = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(acc[c]), 0x100 + D, 0xf, 0xf, false));
    const bool oend = row_down<D>((uint32_t)end) != 0u;
    if (!end && p + D < 16) {
#pragma unroll
        for (int c = 0; c < 16; ++c) acc[c] += o[c];
        end = oend;
    }
}

// ---- paged form ----
// A unit is a block of 1024 samples at one level: every lane works at the same
// level, so its parameters are scalars and the hash products and weights of
// the cluster's cell serve all its evaluations.  Along axis d only the d
// coordinate of an offset evaluation differs from the centre's: one position,
// one comparison and two weights each.  (A sample outside the box has its
// offset points clamped in the other axes too: such lanes are classified by
// whole cells, in the general steps that also take the offsets beyond one
// cell.)
// An emission step puts at most 4 pairs a lane.  Per cluster: the far faces of
// the 6 offset evaluations; their general steps, two each (corners 0-3 or the
// far face, corners 4-7); the centre cell's two.
constexpr int kClusterSteps = 19;   // counted: 6, 6 + 6, 1 (both halves alike)
constexpr int kPairSteps = 2 * kClusterSteps;

__device__ __forceinline__ LevelParams scalar_level(const LevelParams& lp) {
    LevelParams r;
    r.scale = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(lp.scale)));
    r.res = (uint32_t)__builtin_amdgcn_readfirstlane((int)lp.res);
    r.offset = 0u;   // pages hold rows within the level
    r.size_flags = (uint32_t)__builtin_amdgcn_readfirstlane((int)lp.size_flags);
    return r;
}

// One coordinate of an offset evaluation: its cell against the centre's cell
// and its fraction.
__device__ __forceinline__ int offset_cell(const GeoArgs& a, const LevelParams& lp, float base,
                                           bool minus, uint32_t cell, float& frac) {
    const float x = contract1(clampr(base + (minus ? -a.eps : a.eps), a.r), a);
    const float v = __fmaf_rn(lp.scale, x, 0.5f);
    const float fl = floorf(v);
    frac = v - fl;
    return (int)((uint32_t)(int)fl - cell);
}

// A cluster at a level: its centre's cell, and whether the lane's offset
// evaluations must take the general path.
struct ClusterCell {
    LevelPos pos;
    bool general;
};

template <int CL>
__device__ __forceinline__ ClusterCell cluster_cell(const GeoArgs& a, const LevelParams& lp,
                                                    const float P[3]) {
    float xc[3];
    bool out = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        xc[d] = CL == 0 ? contract1(P[d], a) : contract1(clampr(P[d], a.r), a);
        out = out || !(P[d] >= -a.r && P[d] <= a.r);
    }
    return ClusterCell{level_pos(lp, xc), CL == 0 && out};
}

// Corner i (0..3) of the face of a cell with bit `ax` fixed to `b`.
__device__ __forceinline__ int face_corner(int i, int ax, int b) {
    const int low = i & ((1 << ax) - 1);
    return low | (b << ax) | ((i >> ax) << (ax + 1));
}

// Offset evaluation j against the centre's cell by whole cells: `same` cell,
// a face neighbour along `axis` (`adj`; `up`: on its high side), or neither.
struct CellClass {
    LevelPos pos;
    bool same, adj, up;
    int axis;
};

__device__ __forceinline__ CellClass classify(const GeoArgs& a, const LevelParams& lp,
                                              const float P[3], int j, const uint32_t B[3]) {
    float x[3];
    bool inb[3];
    offset_point(a, P, j, x, inb);
    CellClass r;
    r.pos = level_pos(lp, x);
    int nz = 0;
    bool unit = true;
    r.axis = 0;
    r.up = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int dd = (int)(r.pos.c[d] - B[d]);
        if (dd != 0) {
            ++nz;
            r.axis = d;
            r.up = dd > 0;
            unit = unit && (dd == 1 || dd == -1);
        }
    }
    r.same = nz == 0;
    r.adj = nz == 1 && unit;
    return r;
}

// Whether this lane's accumulators start a run of equal cells in its 16 lanes.
__device__ __forceinline__ bool cell_head(const uint32_t B[3], bool live, bool* end) {
    const uint32_t INV = 0xFFFFFFFFu;
    const int p = lane_id() & 15;
    const uint32_t k0 = live ? B[0] : INV, k1 = live ? B[1] : INV, k2 = live ? B[2] : INV;
    if (end) {
        const uint32_t n0 = row_down<1>(k0), n1 = row_down<1>(k1), n2 = row_down<1>(k2);
        *end = (p == 15) || !(n0 == k0 && n1 == k1 && n2 == k2) || k0 == INV;
    }
    const uint32_t u0 = row_up1(k0), u1 = row_up1(k1), u2 = row_up1(k2);
    return live && (p == 0 || !(u0 == k0 && u1 == k1 && u2 == k2));
}

template <int CL>
__device__ __forceinline__ void count_cluster(const GeoArgs& a, const LevelParams& lp,
                                              const float P[3], bool on, bool offsets,
                                              uint32_t* tot) {
    const ClusterCell cc = cluster_cell<CL>(a, lp, P);
    bool touched = CL == 0;
    if (offsets) {
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            float f;
            const int dd = offset_cell(a, lp, P[j >> 1], j & 1, cc.pos.c[j >> 1], f);
            const bool same = !cc.general && dd == 0;
            const bool adj = !cc.general && (dd == 1 || dd == -1);
            touched = touched || same || adj;
            const uint32_t nf = (uint32_t)__popcll(__ballot(on && adj));
            const uint32_t ng = (uint32_t)__popcll(__ballot(on && !cc.general && !same && !adj));
            if (lane_id() == 0) {
                if (nf) atomicAdd(&tot[j], 4u * nf);
                if (ng) {
                    atomicAdd(&tot[6 + j], 4u * ng);
                    atomicAdd(&tot[12 + j], 4u * ng);
                }
            }
        }
        if (CL == 0 && __builtin_expect(__ballot(on && cc.general) != 0, 0)) {
#pragma unroll 1
            for (int j = 0; j < 6; ++j) {
                const CellClass cl = classify(a, lp, P, j, cc.pos.c);
                const bool mine = on && cc.general && !cl.same;
                const uint32_t ng = (uint32_t)__popcll(__ballot(mine && !cl.adj));
                const uint32_t na = (uint32_t)__popcll(__ballot(mine && cl.adj));
                if (lane_id() == 0 && ng + na) {
                    atomicAdd(&tot[6 + j], 4u * (ng + na));
                    atomicAdd(&tot[12 + j], 4u * ng);
                }
            }
        }
    }
    const uint32_t nh =
        (uint32_t)__popcll(__ballot(cell_head(cc.pos.c, on && touched, nullptr)));
    if (lane_id() == 0 && nh) atomicAdd(&tot[18], 4u * nh);
}

// Count pass: per unit (level, block of 1024 samples), the pairs of each
// emission step, from positions alone.  steps[unit][kClusterSteps c + s]:
// cluster c (0: curvature, 1: base and FD), step s (0-5 far faces, 6-11 the
// general evaluations' first halves, 12-17 their second, 18 half the centre
// cell's).  Also keeps the cluster centres
// for the emission.  A block covers levels blockIdx.y, + gridDim.y, ...: all
// of them when the sample blocks alone fill the chip (page_count_split).
__global__ void __launch_bounds__(1024) k_page_count(GeoArgs a, const float* __restrict__ pts,
                                                     const float* __restrict__ randn, int64_t N,
                                                     const float* __restrict__ fdv,
                                                     float* __restrict__ centers,
                                                     uint32_t* __restrict__ steps) {
    __shared__ LevelParams lv[AM_MAX_LEVELS];
    __shared__ uint32_t tot[16 * kPairSteps];
    const int tid = (int)threadIdx.x;
#pragma unroll
    for (int q = 0; q < AM_MAX_LEVELS; ++q)
        if (tid == q && q < a.g.L) lv[q] = a.g.lv[q];
    for (int q = tid; q < 16 * kPairSteps; q += 1024) tot[q] = 0u;
    __syncthreads();
    const int64_t n = (int64_t)blockIdx.x * 1024 + tid;
    const int64_t row = (int64_t)gridDim.x * 1024;
    const bool on = n < N;
    GeoSample s;
    geo_rebuild(a, pts, randn, fdv, n, caller_row(a, n, on), on, s);
    if (blockIdx.y == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            centers[d * row + n] = s.P[d];
            if (a.with_laplace) centers[(3 + d) * row + n] = s.ps[d];
        }
    }
    const bool fd = a.with_grad && !a.analytic;
    for (int l = (int)blockIdx.y; l < a.active; l += (int)gridDim.y) {
        const LevelParams lp = scalar_level(lv[l]);
        if (a.with_laplace) count_cluster<1>(a, lp, s.ps, on, true, tot + l * kPairSteps);
        count_cluster<0>(a, lp, s.P, on, fd, tot + l * kPairSteps + kClusterSteps);
    }
    __syncthreads();
    for (int q = tid; q < a.active * kPairSteps; q += 1024) {
        const int l = q / kPairSteps;
        if (l % (int)gridDim.y == (int)blockIdx.y) steps[((int64_t)l * gridDim.x + blockIdx.x) * kPairSteps + (q - l * kPairSteps)] = tot[q];
    }
}

// Pages and pairs of each unit: the emission's rule (a step that does not fit
// the page any more starts the next one) on the counted steps.
__global__ void k_unit_pages(const uint32_t* __restrict__ steps, int64_t units,
                             uint64_t* __restrict__ out) {
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= units) return;
    uint64_t pages = 0, pairs = 0;
    uint32_t cursor = 0;
    const uint32_t* st = steps + u * kPairSteps;
    for (int c = 0; c < 2; ++c, st += kClusterSteps)
        for (int q = 0; q < 20; ++q) {   // far faces, general halves, centre cell's halves
            const uint32_t n =
                st[q < 6 ? q : (q < 18 ? 6 + ((q & 1) ? 6 : 0) + ((q - 6) >> 1) : 18)];
            if (cursor + n > (uint32_t)kPage) {
                ++pages;
                cursor = 0;
            }
            cursor += n;
            pairs += n;
        }
    if (cursor) ++pages;
    out[u] = pages << 40 | pairs;
}

// Exclusive scan of the units' pages and pairs, and the totals.  One block: a
// unit is 1024 samples of a level, so a thread has few (4.8 M points: 74).
__global__ void __launch_bounds__(1024) k_unit_scan(const uint64_t* __restrict__ in, int64_t units,
                                                    uint64_t* __restrict__ scan,
                                                    int64_t* __restrict__ status) {
    __shared__ uint64_t wave_sum[16];
    const int tid = (int)threadIdx.x;
    const int64_t each = (units + 1023) / 1024;
    const int64_t u0 = tid * each < units ? tid * each : units;
    const int64_t u1 = u0 + each < units ? u0 + each : units;
    uint64_t sum = 0;
    for (int64_t u = u0; u < u1; ++u) sum += in[u];
    uint64_t incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up((unsigned long long)incl, d, 64);
        if ((tid & 63) >= d) incl += o;
    }
    if ((tid & 63) == 63) wave_sum[tid >> 6] = incl;
    __syncthreads();
    uint64_t at = incl - sum, total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        if (w < tid >> 6) at += wave_sum[w];
        total += wave_sum[w];
    }
    for (int64_t u = u0; u < u1; ++u) {
        scan[u] = at;
        at += in[u];
    }
    if (tid == 0) {
        scan[units] = total;
        status[0] = (int64_t)(total >> 40);
        status[1] = 0;
        status[2] = (int64_t)(total & ((1ull << 40) - 1ull));
    }
}

// Emission: one block per unit collects the unit's pairs in an LDS page,
// step by step (all lanes' far faces of one offset evaluation, at most 4096
// pairs), and writes each page partitioned (page_flush).  The counted steps
// say beforehand which steps share a page, so the waves run through them
// without meeting, each taking its place from one LDS counter, and meet only
// to write a page.  Writing pairs straight into partitioned pages spares
// writing them once unpartitioned and reading them back.  LDS (148 KB) holds
// it to one block of 16 waves a CU; bound by VALU issue in the steps and by
// LDS operations in the flushes.  940 k samples, 16 levels, 13 evaluations:
// 2.43 ms, and a forward and backward 11.3 ms, where writing level streams and
// partitioning them in a pass of its own took 13.57 ms.
template <int LJ, class VT>
__global__ void __launch_bounds__(1024) k_pair_pages(GeoArgs a, const float* __restrict__ centers,
                                                     int64_t N, int64_t blocks,
                                                     const float* __restrict__ genc,
                                                     const uint64_t* __restrict__ scan,
                                                     const uint32_t* __restrict__ steps,
                                                     int64_t capacity, uint32_t* __restrict__ keys,
                                                     VT* __restrict__ vals,
                                                     uint16_t* __restrict__ run_start,
                                                     int64_t* __restrict__ status) {
    extern __shared__ char smem[];
    PageLds<VT>& pg = *reinterpret_cast<PageLds<VT>*>(smem);
    const int tid = (int)threadIdx.x, lane = tid & 63, p = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // finest level first
    const int level = a.active - 1 - (int)(blockIdx.x / blocks);
    const int64_t sb = blockIdx.x % blocks;
    const int64_t unit = level * blocks + sb;
    const int64_t page0 = (int64_t)(scan[unit] >> 40);
    const int64_t page_end = (int64_t)(scan[unit + 1] >> 40);
    if (page_end == page0) return;
    if (page_end > capacity) {   // never past the arrays
        for (int64_t q = page0; q < capacity; ++q) page_empty(q, run_start);
        if (tid == 0) status[1] = 1;
        return;
    }
    if (tid <= kMaxDigits) pg.hist[tid] = 0u;
    if (tid == 0) pg.cursor = 0u;
    __shared__ LevelParams lvs;
#pragma unroll
    for (int q = 0; q < AM_MAX_LEVELS; ++q)
        if (q == level && tid == 0) lvs = a.g.lv[q];
    __syncthreads();
    const LevelParams lp = scalar_level(lvs);
    const int64_t n = sb * 1024 + tid, row = blocks * 1024;
    const bool on = n < N;
    int64_t page = page0;
    int cursor = 0;
    const bool spread = (lp.size_flags & kSizeMask) <= (uint32_t)kSpreadDigits * kRows;
    auto flush = [&]() {
        if (page < page_end)
            page_flush(pg, cursor, status + 1, spread, page, keys, vals, run_start);
        else
            __syncthreads();
        ++page;
        cursor = 0;
    };
    const bool hashed = (lp.size_flags & kHashedBit) != 0u;
    const uint32_t my = hashed ? 2654435761u : lp.res, mz = hashed ? 805459861u : lp.res * lp.res;
    // the wave's encode gradients: slot s, feature f at gl[s * LJ * 512 + f * 64 + lane]
    const float* gl = genc + (sb * 16 + wave) * a.genc_slots * (int64_t)(LJ * 512) + level * 128;
    const float* cen = centers + sb * 1024;
    const bool fd = a.with_grad && !a.analytic;

#pragma unroll 1
    for (int c = a.with_laplace ? 0 : 1; c < 2; ++c) {
        const bool curv = c == 0;
        const bool offsets = curv || fd;
        const float* go = gl + (curv ? a.curv0 : 1) * (LJ * 512);   // the offset evaluations
        float P[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) P[d] = on ? (cen + (curv ? 3 + d : d) * row)[tid] : 0.0f;
        ClusterCell cc = curv ? cluster_cell<1>(a, lp, P) : cluster_cell<0>(a, lp, P);
        const uint32_t* B = cc.pos.c;
        float acc[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[q] = 0.0f;
        bool touched = !curv;
        float n0 = 0.0f, n1 = 0.0f;   // the next evaluation's gradients, one ahead
        if (offsets && on) {
            n0 = go[lane];
            n1 = go[64 + lane];
        }
        if (!curv) {   // the base evaluation, always in B
            const float g0 = on ? gl[lane] : 0.0f, g1 = on ? gl[64 + lane] : 0.0f;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float w = corner_weight(cc.pos, t);
                acc[2 * t] = w * g0;
                acc[2 * t + 1] = w * g1;
            }
            // analytic mode: the gradient term u * scale * grad(w_c) . g_x
            if (a.analytic) {
                float ex[3][2];
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
                        ex[d][f] = on ? gl[(a.n_evals + d) * (LJ * 512) + f * 64 + lane] : 0.0f;
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
                        acc[2 * t + f] += (corner_dweight(cc.pos, t, 0) * ex[0][f] +
                                           corner_dweight(cc.pos, t, 1) * ex[1][f]) +
                                          corner_dweight(cc.pos, t, 2) * ex[2][f];
            }
        }
        // per-axis terms of B's corners: lo, and lo plus the axis's factor
        uint32_t lo[3] = {B[0], B[1] * my, B[2] * mz};
        // The cluster's steps, one loop body for all (the unrolled form is
        // larger than the instruction cache): 0-5 the far faces, 6 the general
        // evaluations' halves, 7 and 8 the centre cell's.
        const uint32_t* st = steps + unit * kPairSteps + (curv ? 0 : kClusterSteps);
        // (evaluations with pairs there, and all of a wave with lanes outside the
        // box, whose evaluations may go into B alone)
        uint32_t general = offsets && __ballot(on && cc.general) != 0 ? 63u : 0u;
#pragma unroll
        for (int j = 0; j < 6; ++j) general |= st[6 + j] != 0u ? 1u << j : 0u;
        bool second = false;     // the second half of a general evaluation
        bool head = false;
#pragma unroll 1
        for (int step = offsets ? 0 : 7; step < 9;) {
            // (what derives from these is formed in each step rather than kept in
            // registers across the flushes)
#pragma unroll
            for (int d = 0; d < 3; ++d)
                asm volatile("" : "+v"(cc.pos.f[d]), "+v"(lo[d]), "+v"(P[d]));
            const int gj = __ffs((int)general) - 1;
            const int total = (int)st[step < 6 ? step : (step == 6 ? (second ? 12 : 6) + gj : 18)];
            if (cursor + total > kPage) flush();
            cursor += total;
            // the wave's place in the page for its lanes' four pairs each
            auto place = [&](bool put, uint64_t mask, const uint32_t r[4], const float v[8],
                             uint32_t base) {
                const int n_on = __popcll(mask);
                const int b0 = __builtin_amdgcn_readfirstlane((int)base);
                if (b0 + 4 * n_on > kPage) {   // more than counted
                    if (lane == 0) status[1] = 1;
                } else if (put) {
                    const int at = b0 + (int)__builtin_amdgcn_mbcnt_hi(
                                            (uint32_t)(mask >> 32),
                                            __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        page_put(pg, at + i * n_on, r[i], v[2 * i], v[2 * i + 1]);
                }
            };
            if (__builtin_expect(step == 6, 0)) {   // half a general evaluation
                const CellClass cl = classify(a, lp, P, gj, B);
                const bool in_b = on && cc.general && (cl.same || cl.adj) && !second;
                const bool put = on && ((!cl.same && !cl.adj) || (in_b && cl.adj));
                const float g0 = on ? go[gj * (LJ * 512) + lane] : 0.0f;
                const float g1 = on ? go[gj * (LJ * 512) + 64 + lane] : 0.0f;
                if (in_b) {   // corner t of B: corner t of the cell, or t across the face
                    touched = true;
                    float lo_w[3], hi_w[3];
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const bool flip = cl.adj && cl.axis == d;
                        lo_w[d] = flip ? cl.pos.f[d] : 1.0f - cl.pos.f[d];
                        hi_w[d] = flip ? 1.0f - cl.pos.f[d] : cl.pos.f[d];
                    }
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const float w = ((t & 1 ? hi_w[0] : lo_w[0]) * (t & 2 ? hi_w[1] : lo_w[1])) *
                                        (t & 4 ? hi_w[2] : lo_w[2]);
                        if (cl.same || ((t >> cl.axis) & 1) == (int)cl.up) {
                            acc[2 * t] = __fmaf_rn(w, g0, acc[2 * t]);
                            acc[2 * t + 1] = __fmaf_rn(w, g1, acc[2 * t + 1]);
                        }
                    }
                }
                const uint64_t mask = __ballot(put);
                if (mask != 0) {   // half the cell's 8 corners, or its far face
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(&pg.cursor, (uint32_t)(4 * __popcll(mask)));
                    uint32_t r[4];
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int t = cl.adj ? face_corner(i, cl.axis, cl.up) : (second ? 4 + i : i);
                        r[i] = grid_row(lp, cl.pos.c[0] + (uint32_t)(t & 1),
                                        cl.pos.c[1] + (uint32_t)(t >> 1 & 1),
                                        cl.pos.c[2] + (uint32_t)(t >> 2));
                        const float w = corner_weight(cl.pos, t);
                        v[2 * i] = w * g0;
                        v[2 * i + 1] = w * g1;
                    }
                    place(put, mask, r, v, base);
                }
                if (second) general &= general - 1u;
                second = !second;
                if (general == 0u) step = 7;
                continue;
            }
            // part 1: who puts pairs, and what goes into B
            bool put = false, up = false;
            float wfar[4], g0 = n0, g1 = n1;   // far face: weights and gradients
            if (step < 6) {
                if (step < 5 && on) {
                    n0 = go[(step + 1) * (LJ * 512) + lane];
                    n1 = go[(step + 1) * (LJ * 512) + 64 + lane];
                }
                auto near_faces = [&](auto axis) {
                    constexpr int ax = decltype(axis)::value;
                    constexpr int b = ax == 0 ? 1 : 0, e = ax == 2 ? 1 : 2;   // the other axes
                    float f;
                    const int dd = offset_cell(a, lp, P[ax], (step & 1) != 0, B[ax], f);
                    const bool same = on && !cc.general && dd == 0;
                    put = on && !cc.general && (dd == 1 || dd == -1);
                    touched = touched || same || put;
                    up = dd == 1;
                    // weights of the corners on B's low and high faces (the far
                    // face's are the other face's), as corner_weight forms them
                    const float fl = same ? 1.0f - f : f, fh = same ? f : 1.0f - f;
                    const float fb = cc.pos.f[b], fe = cc.pos.f[e];
                    float wl[4], wh[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float vb = (i & 1) ? fb : 1.0f - fb, ve = (i & 2) ? fe : 1.0f - fe;
                        wl[i] = ax == 2 ? (vb * ve) * fl : (fl * vb) * ve;
                        wh[i] = ax == 2 ? (vb * ve) * fh : (fh * vb) * ve;
                        wfar[i] = up ? wl[i] : wh[i];
                    }
                    if (same || (put && !up)) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = (i & 1) << b | (i >> 1) << e;
                            acc[2 * t] = __fmaf_rn(wl[i], g0, acc[2 * t]);
                            acc[2 * t + 1] = __fmaf_rn(wl[i], g1, acc[2 * t + 1]);
                        }
                    }
                    if (same || (put && up)) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = (i & 1) << b | (i >> 1) << e | 1 << ax;
                            acc[2 * t] = __fmaf_rn(wh[i], g0, acc[2 * t]);
                            acc[2 * t + 1] = __fmaf_rn(wh[i], g1, acc[2 * t + 1]);
                        }
                    }
                };
                if (step < 2) near_faces(std::integral_constant<int, 0>());
                else if (step < 4) near_faces(std::integral_constant<int, 1>());
                else near_faces(std::integral_constant<int, 2>());
            } else {
                // B: equal cells of neighbouring lanes merged, the head emits
                if (step == 7) {
                    bool end;
                    head = cell_head(B, on && touched, &end);
                    merge_step<1>(p, acc, end);
                    merge_step<2>(p, acc, end);
                    merge_step<4>(p, acc, end);
                    merge_step<8>(p, acc, end);
                }
                put = head;
            }
            // part 2: the wave's place in the page, rows and values
            const uint64_t mask = __ballot(put);
            if (mask != 0) {
                uint32_t base = 0;
                if (lane == 0) base = atomicAdd(&pg.cursor, (uint32_t)(4 * __popcll(mask)));
                uint32_t r[4];
                float v[8];
                if (step < 6) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[2 * i] = wfar[i] * g0;
                        v[2 * i + 1] = wfar[i] * g1;
                    }
                    if (step < 2)
                        face_rows(lp, up ? lo[0] + 2u : lo[0] - 1u, lo[1], lo[1] + my, lo[2], lo[2] + mz, r);
                    else if (step < 4)
                        face_rows(lp, up ? lo[1] + 2u * my : lo[1] - my, lo[0], lo[0] + 1u, lo[2],
                                  lo[2] + mz, r);
                    else
                        face_rows(lp, up ? lo[2] + 2u * mz : lo[2] - mz, lo[0], lo[0] + 1u, lo[1],
                                  lo[1] + my, r);
                } else {
                    face_rows(lp, step == 8 ? lo[2] + mz : lo[2], lo[0], lo[0] + 1u, lo[1],
                              lo[1] + my, r);
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = step == 8 ? acc[8 + q] : acc[q];
                }
                place(put, mask, r, v, base);
            }
            if (step < 6) {
                ++step;
                if (step == 6 && general == 0u) step = 7;
            } else {
                ++step;
            }
        }
    }
    if (cursor > 0) flush();
    if (page != page_end) {   // (the page rule on the same steps: not reached)
        for (; page < page_end; ++page) page_empty(page, run_start);
        if (tid == 0) status[1] = 1;
    }
}

// ---- sorted and atomic forms ----
// The pairs of a tile at one level go to [keys, keys + limit): limit is the
// count the count pass found for them; the emit pass makes the same
// decisions, and never writes past limit.  Each lane group (16 lanes, one
// level) has its own.
template <class VT>
struct EmitTile {
    uint32_t* keys;   // the tile's first pair at the level (keys)
    VT* vals;         // the same (values); atomic form: the table gradient
    int cursor;       // group-uniform write position
    int limit;        // pairs reserved
};

// Atomic form (flag "table_atomic"): the "pair array" is the table gradient
// itself, [n_entries] rows of 2 floats, and each pair is added into its row
// with hardware float atomics: no count pass, no sort, no host read, but the
// summation order varies from run to run (the tcnn hash-grid backward's
// semantics).
struct AtomicRow {
    float v[2];
};
template <class VT>
constexpr bool kAtomicPairs = std::is_same<VT, AtomicRow>::value;

// Lanes with `on` write K pairs (rows, values); COUNT only advances the
// cursor.
__device__ __forceinline__ void set_pair(Vals<2>& v, float a, float b) {
    v.v[0] = a;
    v.v[1] = b;
}
__device__ __forceinline__ void set_pair(ValsH<2>& v, float a, float b) {
    v.v[0] = __float2half_rn(a);
    v.v[1] = __float2half_rn(b);
}
__device__ __forceinline__ void set_pair(AtomicRow& v, float a, float b) {   // type-checks only
    v.v[0] = a;
    v.v[1] = b;
}

// The lane group's K * n pairs (n lanes on) fill [cursor, cursor + K n)
// corner-major: pair c of the lane of rank r goes to cursor + c n + r, so each
// store instruction writes consecutive addresses across the group's lanes.
template <int K, bool COUNT, class VT>
__device__ __forceinline__ void emit_pairs(EmitTile<VT>& et, bool on, const uint32_t rows[K],
                                           const float vals[2 * K]) {
    if constexpr (kAtomicPairs<VT>) {
        static_assert(!COUNT, "the atomic form has no count pass");
        if (on) {
#pragma unroll
            for (int c = 0; c < K; ++c) {
                float* row = et.vals[rows[c]].v;
                unsafeAtomicAdd(row, vals[2 * c]);
                unsafeAtomicAdd(row + 1, vals[2 * c + 1]);
            }
        }
        return;
    }
    const int l = lane_id(), k = l >> 4;
    const uint64_t mask = __ballot(on);
    const uint32_t half = (k & 2) ? (uint32_t)(mask >> 32) : (uint32_t)mask;
    const uint32_t group = ((k & 1) ? half >> 16 : half) & 0xffffu;
    const int n_on = __popc(group);
    if (!COUNT && on && et.cursor + K * n_on <= et.limit) {
        const int off = et.cursor + __popc(group & ((1u << (l & 15)) - 1u));
#pragma unroll
        for (int c = 0; c < K; ++c) {
            et.keys[off + c * n_on] = rows[c];
            VT v;
            set_pair(v, vals[2 * c], vals[2 * c + 1]);
            et.vals[off + c * n_on] = v;
        }
    }
    et.cursor += K * n_on;
}

// The 8 corner rows of `cell` at level `lp` (corner c = cell + bits of c).
__device__ __forceinline__ void corner_rows(const LevelParams& lp, const uint32_t cell[3],
                                            uint32_t rows[8]) {
    cell_rows(lp, cell, rows);
}

// Position of cluster evaluation q (0..n-1) for this lane.
template <int CL>
__device__ __forceinline__ void cluster_point(const GeoArgs& a, const GeoSample& s, int q,
                                              float x[3]) {
    bool inb[3];
    if (CL == 0) {  // base, then FD 0..5
        if (q == 0) {
#pragma unroll
            for (int d = 0; d < 3; ++d) x[d] = s.x0[d];
        } else {
            offset_point(a, s.P, q - 1, x, inb);
        }
    } else {        // curvature 0..5
        offset_point(a, s.ps, q, x, inb);
    }
}

// Centre of a cluster: the base point (FD cluster) or the tangent-shifted
// point (curvature cluster; not itself evaluated), clamped and contracted as
// its offsets are.
template <int CL>
__device__ __forceinline__ void cluster_center(const GeoArgs& a, const GeoSample& s, float x[3]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = CL == 0 ? s.x0[d] : contract1(clampr(s.ps[d], a.r), a);
}


// Reduces the stored encode gradients of one cluster of evaluations at level
// slot j into (row, value) pairs with a star-stencil merge.  B = the cell of
// the cluster centre; an evaluation whose cell C
//   * is B adds its 8 corner values into B's accumulators,
//   * is B +- e_axis (a face neighbour, the usual case of an offset of about
//     one cell) adds its 4 corners on the shared face into B's accumulators
//     and emits its 4 far corners,
//   * is anything else emits its 8 corners.
// B's accumulators are then merged with equal-B lanes of the same lane group
// (neighbouring samples of a ray) by a segmented sum in a fixed shuffle
// tree, and the segment head emits them.  Every sum has a fixed order.
// genc_base: this lane's first encode gradient of the tile (genc_lane); the
// cluster's q-th evaluation is genc slot slot0 + q.  COUNT: positions only (no gradients);
// the cursor advances by the lane group's pairs.
template <int LJ, int CL, bool COUNT, class VT>
__device__ __forceinline__ void flush_cluster(const GeoArgs& a, const LevelParams& lp, bool on,
                                              const GeoSample& s, const float* genc_base, int j,
                                              int n_q, int slot0, EmitTile<VT>& et) {
    const int p = lane_id() & 15;
    {
        uint32_t B[3];
        {
            float xc[3];
            cluster_center<CL>(a, s, xc);
            const LevelPos pb = level_pos(lp, xc);
#pragma unroll
            for (int d = 0; d < 3; ++d) B[d] = pb.c[d];
        }
        bool touched = false;
        float acc[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[q] = 0.0f;
        // encode gradients one evaluation ahead: each load pair is issued
        // before the previous evaluation's pair stores, so its latency
        // overlaps that evaluation's work instead of stalling every one
        // (carrying it across level slots too measured no better: more
        // registers)
        float g0n = 0.0f, g1n = 0.0f;
        if constexpr (!COUNT) {
            g0n = genc_base[(slot0 * LJ + j) * 512];
            g1n = genc_base[(slot0 * LJ + j) * 512 + 64];
        }
#pragma unroll 1
        for (int q = 0; q < n_q; ++q) {
            const float g0 = g0n, g1 = g1n;
            if constexpr (!COUNT) {
                if (q + 1 < n_q) {
                    g0n = genc_base[((slot0 + q + 1) * LJ + j) * 512];
                    g1n = genc_base[((slot0 + q + 1) * LJ + j) * 512 + 64];
                }
            }
            float x[3];
            cluster_point<CL>(a, s, q, x);
            const LevelPos pp = level_pos(lp, x);
            // classify C - B
            int ax = -1, sgn = 0, nz = 0;
            bool unit = true;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const int dd = (int)(pp.c[d] - B[d]);
                if (dd != 0) {
                    ++nz;
                    ax = d;
                    sgn = dd;
                    unit = unit && (dd == 1 || dd == -1);
                }
            }
            const bool same = nz == 0;
            const bool adj = nz == 1 && unit;
            const int axm = ax < 0 ? 0 : ax;
            const int far_bit = sgn > 0 ? 1 : 0;  // C's corners off B's face
            touched = touched || same || adj;
            // all 8 corners of C on their own
            {
                const bool em = on && !same && !adj;
                uint32_t rows[8];
                float v[16];
                if (!COUNT && em) corner_rows(lp, pp.c, rows);
                if (!COUNT && em) {
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const float w = corner_weight(pp, c);
                        v[2 * c] = w * g0;
                        v[2 * c + 1] = w * g1;
                    }
                }
                emit_pairs<8, COUNT, VT>(et, em, rows, v);
            }
            // the 4 far corners of a face neighbour
            {
                const bool em = on && adj;
                uint32_t rows[4];
                float v[8];
                if (!COUNT && em) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int c = face_corner(i, axm, far_bit);
                        rows[i] = lp.offset + grid_row(lp, pp.c[0] + (c & 1),
                                                       pp.c[1] + ((c >> 1) & 1),
                                                       pp.c[2] + ((c >> 2) & 1));
                    }
                }
                if (!COUNT && em) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int c = face_corner(i, axm, far_bit);
                        const float w = corner_weight(pp, c);
                        v[2 * i] = w * g0;
                        v[2 * i + 1] = w * g1;
                    }
                }
                emit_pairs<4, COUNT, VT>(et, em, rows, v);
            }
            // into B: corner t of B is corner t of C (same) or corner
            // t ^ (1 << ax) of C when t lies on the shared face (adj)
            if constexpr (!COUNT) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const bool take = same || (adj && ((t >> axm) & 1) == far_bit);
                    const int c = same ? t : (t ^ (1 << axm));
                    const float w = corner_weight(pp, c);
                    if (take) {
                        acc[2 * t] = __fmaf_rn(w, g0, acc[2 * t]);
                        acc[2 * t + 1] = __fmaf_rn(w, g1, acc[2 * t + 1]);
                    }
                }
                // analytic mode, base evaluation (always in B): the gradient
                // term u * scale * grad(w_c) . g_x of each corner
                if (CL == 0 && a.analytic && q == 0) {
                    float ex[3][2];
#pragma unroll
                    for (int d = 0; d < 3; ++d)
#pragma unroll
                        for (int f = 0; f < 2; ++f)
                            ex[d][f] = genc_base[((a.n_evals + d) * LJ + j) * 512 + f * 64];
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
#pragma unroll
                        for (int f = 0; f < 2; ++f) {
                            const float dv = (corner_dweight(pp, t, 0) * ex[0][f] +
                                              corner_dweight(pp, t, 1) * ex[1][f]) +
                                             corner_dweight(pp, t, 2) * ex[2][f];
                            acc[2 * t + f] += dv;
                        }
                    }
                }
            }
        }
        // B: merge equal cells of neighbouring lanes (same lane group),
        // suffix segmented sum in a fixed tree, segment head emits.
        const uint32_t INV = 0xFFFFFFFFu;
        const bool live = on && touched;
        const uint32_t key0 = live ? B[0] : INV, key1 = live ? B[1] : INV,
                       key2 = live ? B[2] : INV;
        const uint32_t n0 = row_down<1>(key0), n1 = row_down<1>(key1), n2 = row_down<1>(key2);
        bool end = (p == 15) || !(n0 == key0 && n1 == key1 && n2 == key2) || key0 == INV;
        if constexpr (!COUNT) {
            merge_step<1>(p, acc, end);
            merge_step<2>(p, acc, end);
            merge_step<4>(p, acc, end);
            merge_step<8>(p, acc, end);
        }
        const uint32_t u0 = row_up1(key0), u1 = row_up1(key1), u2 = row_up1(key2);
        const bool head = live && (p == 0 || !(u0 == key0 && u1 == key1 && u2 == key2));
        uint32_t rows[8];
        if (!COUNT && head) corner_rows(lp, B, rows);
        emit_pairs<8, COUNT, VT>(et, head, rows, acc);
    }
}

// Pair pass.  COUNT: the number of (row, value) pairs each tile of 16
// samples emits at each level, from positions alone (counts[level * tiles +
// tile]).  Otherwise: the same decisions with the encode gradients, the pairs
// written from offsets[level * tiles + tile] on (one stream per level, never
// past the tile's count; a different count sets status[1]).
template <int LJ, bool COUNT, class VT>
__global__ void __launch_bounds__(256) k_geo_pairs(
    GeoArgs a, const float* __restrict__ pts, const float* __restrict__ randn, int64_t N,
    const float* __restrict__ fdv, const float* __restrict__ genc, uint32_t* __restrict__ keys,
    VT* __restrict__ vals, const int64_t* __restrict__ offsets, int64_t* __restrict__ counts,
    int64_t* __restrict__ status, int64_t capacity) {
    __shared__ LevelParams lv[AM_MAX_LEVELS];
#pragma unroll
    for (int q = 0; q < AM_MAX_LEVELS; ++q)
        if ((int)threadIdx.x == q && q < a.g.L) lv[q] = a.g.lv[q];
    __syncthreads();
    const int l = lane_id(), p = l & 15, k = l >> 4;
    const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6;
    const int64_t n_tiles = (N + 15) / 16;
    for (int64_t tile = (int64_t)blockIdx.x * nw + wave; tile < n_tiles;
         tile += (int64_t)gridDim.x * nw) {
        const int64_t n = tile * 16 + p;
        const bool valid = n < N;
        GeoSample s;
        geo_rebuild(a, pts, randn, fdv, n, caller_row(a, n, valid), valid, s);
        const float* gt = COUNT ? nullptr : genc + genc_lane(a, tile, LJ, l);
#pragma unroll 1
        for (int j = 0; j < LJ; ++j) {
            const int level = k + 4 * j;
            const bool there = level < a.g.L;
            const bool on = valid && level < a.active;
            const int64_t entry = level * n_tiles + tile;
            LevelParams lp{};
            if (there) lp = lv[level];
            EmitTile<VT> et{nullptr, nullptr, 0, 0};
            if constexpr (kAtomicPairs<VT>) {
                et.vals = vals;
            } else if constexpr (!COUNT) {
                if (there) {
                    const int64_t off = offsets[entry];
                    const int64_t room = capacity - off;
                    int64_t lim = counts[entry];
                    if (lim > room) {   // cut at the arrays' capacity, flagged
                        lim = room > 0 ? room : 0;
                        if (p == 0) status[1] = 1;
                    }
                    et = EmitTile<VT>{keys + off, vals + off, 0, (int)lim};
                }
            }
            if (a.with_laplace)
                flush_cluster<LJ, 1, COUNT>(a, lp, on, s, gt, j, 6, a.curv0, et);
            flush_cluster<LJ, 0, COUNT>(a, lp, on, s, gt, j, a.with_grad && !a.analytic ? 7 : 1, 0,
                                        et);
            if constexpr (COUNT) {
                if (there && p == 0) counts[entry] = et.cursor;
            } else if constexpr (!kAtomicPairs<VT>) {
                if (there && p == 0 && et.cursor != et.limit) status[1] = 1;
            }
        }
    }
}

// Sentinel keys and zero values in [status[0], bound): the unused tail of
// pair arrays carved for the worst-case bound (sorted form).
template <class VT>
__global__ void k_pair_tail(uint32_t* __restrict__ keys, VT* __restrict__ vals,
                            const int64_t* __restrict__ status, int64_t bound, uint32_t sentinel) {
    const int64_t first = status[0];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = first + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < bound;
         i += stride) {
        keys[i] = sentinel;
        VT v;
        set_pair(v, 0.0f, 0.0f);
        vals[i] = v;
    }
}

// status[0] = status[2] = number of pairs; status[1] = 0, set by the emit pass
// on a count mismatch.
__global__ void k_pair_total(const int64_t* __restrict__ offsets,
                             const int64_t* __restrict__ counts, int64_t entries,
                             int64_t* __restrict__ status) {
    if (threadIdx.x == 0) {
        const int64_t n = offsets[entries - 1] + counts[entries - 1];
        status[0] = n;
        status[1] = 0;
        status[2] = n;
    }
}

// ---- host side ----
// Most pairs a sample's lane can emit at one level.  FD cluster: the base
// point is always in B, so 6 x 8 + 8 for B = 56; analytic or without
// gradient: the base alone, 8.  Curvature cluster (its centre is not
// evaluated): 6 x 8 = 48 with B untouched; with one point in a face
// neighbour of B, 5 x 8 + 4 far corners + 8 for B = 52 (the most); more
// points in or beside B emit less.
static int64_t lane_pairs(const GeoArgs& a) {
    return (a.with_grad && !a.analytic ? 56 : 8) + (a.with_laplace ? 52 : 0);
}

void pairs_carve(WsCarver& c, const GeoArgs& a, const am_grid_desc* g, int64_t n, PairHead* out) {
    PairHead h{};
    h.paged = table_paged(g);
    h.status = c.take<int64_t>(4);
    if (h.paged) {
        const int64_t blocks = ceil_div(n, 1024);
        h.units = blocks * a.active;
        h.centers = c.take<float>((size_t)blocks * 1024 * 6);
        h.steps = c.take<uint32_t>((size_t)h.units * kPairSteps + 1);
        h.unit_pages = c.take<uint64_t>((size_t)h.units + 1);
        h.unit_scan = c.take<uint64_t>((size_t)h.units + 1);
    } else {
        size_t sb = 0;
        h.entries = ceil_div(n, 16) * a.g.L;
        h.counts = c.take<int64_t>((size_t)h.entries + 1);
        h.offsets = c.take<int64_t>((size_t)h.entries + 1);
        rocprim::exclusive_scan(nullptr, sb, (const int64_t*)nullptr, (int64_t*)nullptr, (int64_t)0,
                                (size_t)(h.entries > 0 ? h.entries : 1), rocprim::plus<int64_t>(),
                                0, false);
        h.scan_bytes = sb;
        h.scan_tmp = c.take<char>(sb + 256);
    }
    *out = h;
}

// A step that does not fit leaves less than 4096 pairs' room in its page.
int64_t pairs_bound(const GeoArgs& a, const PairHead& h, int LJ, int64_t n) {
    if (!h.paged) return ceil_div(n, 16) * (lane_pairs(a) * LJ * 64);
    auto pages = [&](int64_t samples) { return lane_pairs(a) * samples / (kPage - 4096) + 1; };
    const int64_t whole = n / 1024, rest = n % 1024;   // units of 1024 samples, and a smaller one
    return a.active * (whole * pages(1024) + (rest ? pages(rest) : 0));
}

// Moves one count (flag "sdf_bwd_count_shift"), so that a test can see the
// emission's check of the counts.  The emission never passes its page's end,
// however many pairs were counted.
__global__ void k_shift_count(uint32_t* count, int by) {
    const int c = (int)*count + by;
    *count = c < 0 ? 0u : (uint32_t)c;
}

static int shift_count(uint32_t* count, hipStream_t s) {
    const int by = flag_value("sdf_bwd_count_shift", 0);
    if (by == 0) return AM_OK;
    AM_CHECK_ARG(by >= -64 && by <= 64, "sdf_bwd_count_shift %d", by);
    hipLaunchKernelGGL(k_shift_count, dim3(1), dim3(1), 0, s, count, by);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <int LJ>
static void count_launch(const GeoArgs& a, const float* pts, const float* randn, int64_t n,
                         const float* fdv, int64_t* counts, hipStream_t s) {
    hipLaunchKernelGGL((k_geo_pairs<LJ, true, Vals<2>>), dim3(count_blocks(n)), dim3(256), 0, s, a,
                       pts, randn, n, fdv, nullptr, nullptr, nullptr, nullptr, counts, nullptr,
                       (int64_t)0);
}

// Few sample blocks leave the chip idle: their levels are split over blocks
// until there are two a CU (20 k samples: 49 -> 15 us; 65 k: 29 -> 14 us; at
// 940 k, where nothing is split, 150 us).
static unsigned page_count_split(int64_t blocks, int active) {
    const int64_t want = ceil_div(512, blocks);
    return (unsigned)(want < 1 ? 1 : (want > active ? (active > 0 ? active : 1) : want));
}

int pairs_count(const GeoArgs& a, int LJ, const float* pts, const float* randn, int64_t n,
                const float* fdv, PairHead& h, hipStream_t s) {
    KernelTimer kt_("pair_count", s);
    if (h.paged) {
        const int64_t blocks = ceil_div(n, 1024);
        if (blocks > 0) {
            hipLaunchKernelGGL(k_page_count, dim3((unsigned)blocks, page_count_split(blocks, a.active)),
                               dim3(1024), 0, s, a, pts, randn, n, fdv, h.centers, h.steps);
            AM_LAUNCH_CHECK();
        }
        if (h.units > 0) {
            // (the base cluster's centre cells of the first unit)
            if (int rc = shift_count(h.steps + 2 * kClusterSteps - 1, s)) return rc;
            hipLaunchKernelGGL(k_unit_pages, dim3((unsigned)ceil_div(h.units, 256)), dim3(256), 0, s,
                               h.steps, h.units, h.unit_pages);
            AM_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(k_unit_scan, dim3(1), dim3(1024), 0, s, h.unit_pages, h.units,
                           h.unit_scan, h.status);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    if (LJ == 2) count_launch<2>(a, pts, randn, n, fdv, h.counts, s);
    else count_launch<4>(a, pts, randn, n, fdv, h.counts, s);
    AM_LAUNCH_CHECK();
    size_t sb = h.scan_bytes;
    hipError_t e = rocprim::exclusive_scan(h.scan_tmp, sb, h.counts, h.offsets, (int64_t)0,
                                           (size_t)h.entries, rocprim::plus<int64_t>(), s, false);
    if (e != hipSuccess) {
        set_error("pair-count scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    hipLaunchKernelGGL(k_pair_total, dim3(1), dim3(64), 0, s, h.offsets, h.counts, h.entries,
                       h.status);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <int LJ, class VT>
static int pages_launch(const GeoArgs& a, int64_t n, const float* genc, PairHead& h, TablePages& tp,
                        hipStream_t s) {
    auto kern = k_pair_pages<LJ, VT>;
    AM_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sizeof(PageLds<VT>)));
    KernelTimer kt_("pair_emit", s);
    hipLaunchKernelGGL(kern, dim3((unsigned)h.units), dim3(kPageThreads), sizeof(PageLds<VT>), s, a,
                       h.centers, n, ceil_div(n, 1024), genc, h.unit_scan, h.steps, tp.pages, tp.keys,
                       reinterpret_cast<VT*>(tp.vals), tp.run_start, h.status);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <int LJ, class V>
static int arrays_launch(const GeoArgs& a, const float* pts, const float* randn, int64_t n,
                         const float* fdv, const float* genc, PairHead& h, TableReduceWs& tw,
                         bool bounded, hipStream_t s) {
    if (bounded && tw.m > 0) {   // the arrays' unused tail
        const int64_t want = ceil_div(tw.m, 256);
        hipLaunchKernelGGL((k_pair_tail<V>), dim3((unsigned)(want < 16384 ? want : 16384)), dim3(256),
                           0, s, tw.keys[0], reinterpret_cast<V*>(tw.vals[0]), h.status, tw.m,
                           table_sentinel(tw.end_bit));
        AM_LAUNCH_CHECK();
    }
    KernelTimer kt_("pair_emit", s);
    hipLaunchKernelGGL((k_geo_pairs<LJ, false, V>), dim3(pair_blocks(n)), dim3(256), 0, s, a, pts,
                       randn, n, fdv, genc, tw.keys[0], reinterpret_cast<V*>(tw.vals[0]), h.offsets,
                       h.counts, h.status, tw.m);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

int pairs_reduce(const GeoArgs& a, int LJ, const am_grid_desc* g, const float* pts,
                 const float* randn, int64_t n, const float* fdv, const float* genc, PairHead& h,
                 TablePages& tp, TableReduceWs& tw, bool bounded, float* dtable, hipStream_t s) {
    const bool half = a.prec == AM_PREC_MIXED;
    int rc = AM_OK;
    if (!h.paged) {
        if (half)
            rc = LJ == 2 ? arrays_launch<2, ValsH<2>>(a, pts, randn, n, fdv, genc, h, tw, bounded, s)
                         : arrays_launch<4, ValsH<2>>(a, pts, randn, n, fdv, genc, h, tw, bounded, s);
        else
            rc = LJ == 2 ? arrays_launch<2, Vals<2>>(a, pts, randn, n, fdv, genc, h, tw, bounded, s)
                         : arrays_launch<4, Vals<2>>(a, pts, randn, n, fdv, genc, h, tw, bounded, s);
        return rc ? rc : table_reduce_run(tw, g, dtable, s);
    }
    if (h.units > 0) {
        if (half)
            rc = LJ == 2 ? pages_launch<2, uint32_t>(a, n, genc, h, tp, s)
                         : pages_launch<4, uint32_t>(a, n, genc, h, tp, s);
        else
            rc = LJ == 2 ? pages_launch<2, uint2>(a, n, genc, h, tp, s)
                         : pages_launch<4, uint2>(a, n, genc, h, tp, s);
        if (rc) return rc;
    }
    return table_pages_run(tp, g, h.unit_scan, ceil_div(n, 1024), a.active, 0, dtable, s);
}

int pairs_atomic(const GeoArgs& a, int LJ, const float* pts, const float* randn, int64_t n,
                 const float* fdv, const float* genc, float* dtable, hipStream_t s) {
    KernelTimer kt_("pair_atomic", s);
    auto kern = LJ == 2 ? k_geo_pairs<2, false, AtomicRow> : k_geo_pairs<4, false, AtomicRow>;
    hipLaunchKernelGGL(kern, dim3(pair_blocks(n)), dim3(256), 0, s, a, pts, randn, n, fdv, genc,
                       nullptr, reinterpret_cast<AtomicRow*>(dtable), nullptr, nullptr, nullptr,
                       (int64_t)0);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

}  // namespace am
