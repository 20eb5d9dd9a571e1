// Ray-AABB intersection and occupancy-grid ray marching (nerfacc 0.3.3
// ray_aabb_intersect + ray_marching with AABB contraction and cone angle 0,
// as called at models/neus.py:209-220): count pass -> exclusive scan ->
// fill pass, giving packed ray-sorted (ray_indices, t_starts, t_ends).
//
// The arithmetic is the same IEEE sequence as the C restatement in the
// oracle (built with -ffp-contract=off; `origin + t_mid*dir` fused), so
// sample intervals and ray indices are bit-exact with it.  Build-side
// additions shared with the oracle: an optional per-ray sample cap and the
// end of a ray when a step no longer advances t.
#include <cmath>
#include <rocprim/device/device_scan.hpp>
#include "am_common.h"

namespace am {

struct MarchArgs {
    float roi[6];
    int res;
    float step;
    int cap;
    int has_grid;
    // Division by a power of two is an exact scaling, so x / range and
    // x * (1 / range) are the same IEEE result: the divisions of the marching
    // rule become multiplications where the roi extent (and the grid
    // resolution) is a power of two, as for the usual [-r, r]^3 with r = 2^k.
    float inv_range[3];
    int range_pow2;  // bit d: roi extent of axis d is a power of two
    float inv_res;
    int res_pow2;
};

__device__ __forceinline__ float div_range(const MarchArgs& a, float x, int d) {
    return ((a.range_pow2 >> d) & 1) ? x * a.inv_range[d] : x / (a.roi[3 + d] - a.roi[d]);
}

__device__ __forceinline__ float div_res(const MarchArgs& a, float x) {
    return a.res_pow2 ? x * a.inv_res : x / (float)a.res;
}

__device__ __forceinline__ void aabb_one(const float* o, const float* d, const float* aabb,
                                         float* t_near, float* t_far) {
    float tmin = (aabb[0] - o[0]) / d[0];
    float tmax = (aabb[3] - o[0]) / d[0];
    if (tmin > tmax) { const float t = tmin; tmin = tmax; tmax = t; }
    float tymin = (aabb[1] - o[1]) / d[1];
    float tymax = (aabb[4] - o[1]) / d[1];
    if (tymin > tymax) { const float t = tymin; tymin = tymax; tymax = t; }
    if (tmin > tymax || tymin > tmax) { *t_near = 1e10f; *t_far = 1e10f; return; }
    if (tymin > tmin) tmin = tymin;
    if (tymax < tmax) tmax = tymax;
    float tzmin = (aabb[2] - o[2]) / d[2];
    float tzmax = (aabb[5] - o[2]) / d[2];
    if (tzmin > tzmax) { const float t = tzmin; tzmin = tzmax; tzmax = t; }
    if (tmin > tzmax || tzmin > tmax) { *t_near = 1e10f; *t_far = 1e10f; return; }
    if (tzmin > tmin) tmin = tzmin;
    if (tzmax < tmax) tmax = tzmax;
    *t_near = tmin > 0.0f ? tmin : 0.0f;
    *t_far = tmax;
}

__device__ __forceinline__ bool occupied(const MarchArgs& a, const float xyz[3],
                                         const uint8_t* __restrict__ grid) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (xyz[d] < a.roi[d] || xyz[d] > a.roi[3 + d]) return false;
    if (!a.has_grid) return true;
    int ix[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float u = div_range(a, xyz[d] - a.roi[d], d);
        int v = (int)(u * (float)a.res);
        v = v < 0 ? 0 : (v > a.res - 1 ? a.res - 1 : v);
        ix[d] = v;
    }
    return grid[((int64_t)ix[0] * a.res + ix[1]) * a.res + ix[2]] != 0;
}

__device__ __forceinline__ float dist_next_voxel(const MarchArgs& a, const float xyz[3],
                                                 const float dir[3], const float inv[3]) {
    float t = INFINITY;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float range = a.roi[3 + d] - a.roi[d];
        const float u = div_range(a, xyz[d] - a.roi[d], d) * (float)a.res;
        const float sg = copysignf(1.0f, dir[d]);
        const float tt = div_res(a, (floorf(u + 0.5f + 0.5f * sg) - u) * inv[d]) * range;
        t = fminf(t, tt);
    }
    return fmaxf(t, 0.0f);
}

// ---- marching, a wave to a ray ----
// The rule for one ray (nerfacc 0.3.3): from t0 = near, t1 = t0 + step,
// t_mid = (t0 + t1) / 2, while t_mid < far and fewer than cap samples (cap 0:
// no cap): the midpoint's cell occupied -> a sample [t0, t1], then t0 = t1,
// t1 = t0 + step, t_mid = (t0 + t1) / 2, and the ray ends when t_mid no
// longer grows; unoccupied -> t_mid advances by whole steps to the next voxel
// boundary (the ray ends when a step no longer advances t), t0 / t1 = t_mid
// -/+ step / 2.
// A wave runs it, so the grid loads of up to 64 points are in flight together
// instead of one after another.  A round takes one of two forms, from the
// state (t0, t1, t_mid, j):
//   * inside: lane g takes g occupied steps and tests its midpoint.  The first
//     lane whose state is out of range or unoccupied ends the run: the lanes
//     before it are the next samples; if it is in range, the march goes on
//     outside from its midpoint.
//   * outside: the midpoints of a run of voxel skips all lie on the sequence
//     s_0 = t_mid, s_k+1 = s_k + step.  Lane g holds s_g, tests it, and finds
//     from its own skip target where the skip from s_g lands (`next`); the
//     chain of skips from s_0 is then followed through the lanes, to the first
//     midpoint that is occupied (inside from there), out of range or stuck (the
//     ray ends), or whose skip leaves the lanes (the next round starts where it
//     lands).
// Both need the sequence x_0, x_k+1 = fl(x_k + step), and every lane its
// element at once: within a binade an addition moves by the same d = fl(x_0 +
// step) - x_0 (but for a tie), so lane k proposes fl(x_0 + k d), checks that
// fl(its element + step) is the next lane's, and the round uses the lanes up to
// the first that disagrees (one lane at least).
// Samples and counts are those of the one-lane rule, bit for bit.  Outputs
// ts / te / ri may be null (count only); every lane returns the count.
// Latency-bound: a chain of rounds, a grid load and some hundred instructions
// each, with few waves a CU.  2048 rays, 128^3 cells, steps of 0.43 cell: 43 us;
// 16 lanes a ray, serial sequences: 141 us; 4 lanes and one skip a round: 355 us
// (whole marching call with 256 / 8192 / 262144 rays: 45 / 91 / 695 us, against
// 182 / 307 / 910 with 4 lanes).
__device__ __forceinline__ float lane_float(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ int march_wave(const MarchArgs& a, const float* o, const float* d,
                                          float near, float far,
                                          const uint8_t* __restrict__ grid,
                                          float* __restrict__ ts, float* __restrict__ te,
                                          int32_t* __restrict__ ri, int32_t ray) {
    const int g = lane_id();
    const float fg = (float)g;
    const float inv[3] = {1.0f / d[0], 1.0f / d[1], 1.0f / d[2]};
    const float step = a.step, inv_step = 1.0f / step;
    float t0 = near;
    float t1 = t0 + step;
    float tm = (t0 + t1) * 0.5f;
    int j = 0;
    bool inside = true;
    while (true) {
        // this lane's element x of the sequence from t1 (inside: the end of its
        // interval) or from t_mid, its predecessors, and the lanes that hold
        const float base = inside ? t1 : tm;
        const float delta = (base + step) - base;
        const float x = __fmaf_rn(fg, delta, base);
        const uint64_t agree = __ballot(x + step == __fmaf_rn(fg + 1.0f, delta, base));
        const int hold = ~agree == 0 ? 64 : min(__builtin_ctzll(~agree) + 1, 64);
        const float x1 = __fmaf_rn(fg - 1.0f, delta, base), x2 = __fmaf_rn(fg - 2.0f, delta, base);
        const float c0 = g == 0 ? t0 : x1;
        const float cm = !inside ? x : (g == 0 ? tm : (x1 + x) * 0.5f);
        const bool alive = !inside || g == 0 || cm > (g == 1 ? tm : (x2 + x1) * 0.5f);
        const bool cond = g < hold && alive && cm < far &&
                          !(a.cap > 0 && j + (inside ? g : 0) >= a.cap);
        float xyz[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) xyz[k] = __fmaf_rn(cm, d[k], o[k]);
        const bool occ = cond && occupied(a, xyz, grid);
        const uint64_t bo = __ballot(occ);
        if (inside) {
            // first lane that is not an occupied in-range state
            const int m = ~bo == 0 ? 64 : __builtin_ctzll(~bo);
            if (g < m && ts) {
                ts[j + g] = c0;
                te[j + g] = x;
                if (ri) ri[j + g] = ray;
            }
            j += m;
            if (m == hold) {   // all were samples: on from the last lane's successor
                t0 = lane_float(x, hold - 1);
                t1 = t0 + step;
                tm = (t0 + t1) * 0.5f;
                if (!(tm > lane_float(cm, hold - 1))) break;
                continue;
            }
            if (!(__ballot(cond) >> m & 1u)) break;   // state m ends the march
            // state m is in range and unoccupied: voxel skips from its midpoint
            tm = lane_float(cm, m);
            inside = false;
            continue;
        }
        const float goal = x + dist_next_voxel(a, xyz, d, inv);
        // the first element after x not below goal: about where it is, then exactly
        int next = g + max(1, (int)fminf((goal - x) * inv_step, 64.0f));
        while (next > g + 1 && !(__fmaf_rn((float)(next - 1), delta, base) < goal)) --next;
        while (next < 64 && __fmaf_rn((float)next, delta, base) < goal) ++next;
        // 0: skips to lane `next`; 1: occupied; 2: the ray ends; 3: skips past the lanes
        const int kind = occ ? 1 : (!cond || !(x + step > x) ? 2 : (next < hold ? 0 : 3));
        int hop = kind == 0 ? next : g;
#pragma unroll
        for (int q = 0; q < 6; ++q) hop = __shfl(hop, hop, 64);   // 64 skips
        const int last = __builtin_amdgcn_readfirstlane(hop);
        const int end = __builtin_amdgcn_readlane(kind, last);
        if (end == 2) break;
        if (end == 1) {
            tm = lane_float(x, last);
            t0 = tm - step * 0.5f;
            t1 = tm + step * 0.5f;
            inside = true;
        } else {
            // from the last element: below the target, or the skip's start
            const float target = lane_float(goal, last);
            float tt = lane_float(x, hold - 1);
            bool stuck = false;
            do {
                const float nt = tt + step;
                if (!(nt > tt)) {
                    stuck = true;
                    break;
                }
                tt = nt;
            } while (tt < target);
            if (stuck) break;
            tm = tt;
        }
    }
    return j;
}

// Lanes per ray of march_group and of the background marching (8 measured no
// faster).
constexpr int kMarchGroup = 4;

// The same with kMarchGroup lanes to a ray, for many rays of few steps or of
// many steps a cell, where a wave to a ray leaves most of its lanes idle or
// within few cells (use_group): inside, the
// group's lanes take their steps as above but by the additions themselves;
// a voxel skip is walked from the first lane outside.
__device__ int march_group(const MarchArgs& a, const float* o, const float* d, float near,
                           float far, const uint8_t* __restrict__ grid, float* __restrict__ ts,
                           float* __restrict__ te, int32_t* __restrict__ ri, int32_t ray) {
    constexpr int G = kMarchGroup;
    const int g = lane_id() % G, gbase = lane_id() - g;
    const float inv[3] = {1.0f / d[0], 1.0f / d[1], 1.0f / d[2]};
    const float step = a.step;
    const uint32_t mask = (1u << G) - 1u;
    float t0 = near;
    float t1 = t0 + step;
    float tm = (t0 + t1) * 0.5f;
    int j = 0;
    while (true) {
        // this lane's state: g occupied steps ahead
        float c0 = t0, c1 = t1, cm = tm;
        bool alive = true;
        for (int q = 0; q < g; ++q) {
            const float prev = cm;
            c0 = c1;
            c1 = c0 + step;
            cm = (c0 + c1) * 0.5f;
            alive = alive && (cm > prev);
        }
        const bool cond = alive && cm < far && !(a.cap > 0 && j + g >= a.cap);
        float xyz[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) xyz[k] = __fmaf_rn(cm, d[k], o[k]);
        const bool occ = cond && occupied(a, xyz, grid);
        const uint32_t bo = (uint32_t)(__ballot(occ) >> gbase) & mask;
        const uint32_t bc = (uint32_t)(__ballot(cond) >> gbase) & mask;
        const int m = __builtin_ctz(~bo);   // first lane not an occupied in-range state (G: none)
        if (g < m && ts) {
            ts[j + g] = c0;
            te[j + g] = c1;
            if (ri) ri[j + g] = ray;
        }
        if (m == G) {   // all G were samples: continue from the last lane's successor
            const float n0 = c1, n1 = n0 + step, nm = (n0 + n1) * 0.5f;
            const int ok = nm > cm ? 1 : 0;
            t0 = __shfl(n0, gbase + G - 1, 64);
            t1 = __shfl(n1, gbase + G - 1, 64);
            tm = __shfl(nm, gbase + G - 1, 64);
            const int okg = __shfl(ok, gbase + G - 1, 64);
            j += G;
            if (!okg) break;
            continue;
        }
        j += m;
        if (!((bc >> m) & 1u)) break;   // state m ends the march
        // state m is in range and unoccupied: the voxel skip from its midpoint
        const float tmm = __shfl(cm, gbase + m, 64);
#pragma unroll
        for (int k = 0; k < 3; ++k) xyz[k] = __fmaf_rn(tmm, d[k], o[k]);
        const float target = tmm + dist_next_voxel(a, xyz, d, inv);
        float tt = tmm;
        bool stuck = false;
        do {
            const float nt = tt + step;
            if (!(nt > tt)) {
                stuck = true;
                break;
            }
            tt = nt;
        } while (tt < target);
        if (stuck) break;
        tm = tt;
        t0 = tm - step * 0.5f;
        t1 = tm + step * 0.5f;
    }
    return j;
}

// Ray and lane of a thread of the marching kernels: four waves or (GROUP) 64
// groups of lanes a block.
template <bool GROUP>
__device__ __forceinline__ int64_t march_ray() {
    if constexpr (GROUP) return ((int64_t)blockIdx.x * 256 + threadIdx.x) / kMarchGroup;
    else return (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
}
template <bool GROUP>
__device__ __forceinline__ int march(const MarchArgs& a, const float* o, const float* d, float near,
                                     float far, const uint8_t* __restrict__ grid,
                                     float* __restrict__ ts, float* __restrict__ te,
                                     int32_t* __restrict__ ri, int32_t ray) {
    if constexpr (GROUP) return march_group(a, o, d, near, far, grid, ts, te, ri, ray);
    else return march_wave(a, o, d, near, far, grid, ts, te, ri, ray);
}
template <bool GROUP>
__device__ __forceinline__ bool march_lead() {
    return lane_id() % (GROUP ? kMarchGroup : 64) == 0;
}

// ---- background marching (nerfacc 0.3.3 ray_marching with
// ContractionType.UN_BOUNDED_SPHERE and a cone angle, as called by
// models/neus.py:141-171): steps of dt = clamp(t0 * cone, step, 1e10), a
// sample kept when its midpoint's cell of the contracted grid is occupied;
// contracted scenes take no voxel skip.  [near, far] per ray come from the
// caller (its near/far planes and stratified jitter). ----
struct MarchBgArgs {
    MarchArgs m;
    float cone;
};

// Unbounded-sphere contraction of a world point into [0, 1]^3: unit cube of
// the roi -> [-1, 1]; |x| > 1 maps to (2 - 1/|x|) x/|x|; then x/4 + 1/2.
__device__ __forceinline__ bool occupied_unbounded(const MarchArgs& a, const float xyz[3],
                                                   const uint8_t* __restrict__ grid) {
    if (!a.has_grid) return true;
    float x[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = div_range(a, xyz[d] - a.roi[d], d) * 2.0f - 1.0f;
    const float mag = sqrtf((x[0] * x[0] + x[1] * x[1]) + x[2] * x[2]);
    if (mag > 1.0f) {
        const float k = 2.0f - 1.0f / mag;
#pragma unroll
        for (int d = 0; d < 3; ++d) x[d] = k * (x[d] / mag);
    }
    int ix[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float u = x[d] * 0.25f + 0.5f;
        int v = (int)(u * (float)a.res);
        v = v < 0 ? 0 : (v > a.res - 1 ? a.res - 1 : v);
        ix[d] = v;
    }
    return grid[((int64_t)ix[0] * a.res + ix[1]) * a.res + ix[2]] != 0;
}

__device__ __forceinline__ float cone_dt(const MarchBgArgs& b, float t) {
    return fminf(fmaxf(t * b.cone, b.m.step), 1e10f);
}

// The background rule: from t0 = near, t1 = t0 + dt(t0), while t_mid < far
// and fewer than cap samples: the midpoint's contracted cell occupied -> a
// sample [t0, t1]; then t0 = t1, t1 = t0 + dt(t0), and the ray ends when
// t_mid no longer grows.  The steps do not depend on occupancy, so G lanes
// take G steps a round: lane g's state is g steps ahead, its sample index j
// plus the occupied lanes before it; the first state out of range (or at
// the cap) ends the ray.  Bit-exact with the one-lane rule.
template <int G>
__device__ int march_group_bg(const MarchBgArgs& b, const float* o, const float* d, float near,
                              float far, const uint8_t* __restrict__ grid, float* __restrict__ ts,
                              float* __restrict__ te, int32_t* __restrict__ ri, int32_t ray,
                              int g, int gbase) {
    const uint32_t mask = (1u << G) - 1u;
    float t0 = near;
    float t1 = t0 + cone_dt(b, t0);
    float tm = (t0 + t1) * 0.5f;
    int j = 0;
    while (true) {
        float c0 = t0, c1 = t1, cm = tm;
        bool alive = true;
        for (int q = 0; q < g; ++q) {
            const float prev = cm;
            c0 = c1;
            c1 = c0 + cone_dt(b, c0);
            cm = (c0 + c1) * 0.5f;
            alive = alive && (cm > prev);
        }
        const bool valid = alive && cm < far;
        float xyz[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) xyz[k] = __fmaf_rn(cm, d[k], o[k]);
        const bool occ = valid && occupied_unbounded(b.m, xyz, grid);
        const uint32_t bo = (uint32_t)(__ballot(occ) >> gbase) & mask;
        const int jg = j + __builtin_popcount(bo & ((1u << g) - 1u));   // this state's index
        const bool ends = !valid || (b.m.cap > 0 && jg >= b.m.cap);
        const uint32_t be = (uint32_t)(__ballot(ends) >> gbase) & mask;
        const int e = be ? __builtin_ctz(be) : G;   // first state that ends the ray
        if (g < e && occ && ts) {
            ts[jg] = c0;
            te[jg] = c1;
            ri[jg] = ray;
        }
        j += __builtin_popcount(bo & (e == G ? mask : ((1u << e) - 1u)));
        if (e < G) break;
        const float n0 = c1, n1 = n0 + cone_dt(b, n0), nm = (n0 + n1) * 0.5f;
        const int ok = nm > cm ? 1 : 0;
        t0 = __shfl(n0, gbase + G - 1, 64);
        t1 = __shfl(n1, gbase + G - 1, 64);
        tm = __shfl(nm, gbase + G - 1, 64);
        if (!__shfl(ok, gbase + G - 1, 64)) break;
    }
    return j;
}

// G lanes to a ray (whole groups share a ray and exit together).
__global__ void __launch_bounds__(64) k_march_bg_count(MarchBgArgs b,
                                                      const float* __restrict__ rays, int64_t n,
                                                      const float* __restrict__ t_near,
                                                      const float* __restrict__ t_far,
                                                      const uint8_t* __restrict__ grid,
                                                      int32_t* __restrict__ counts) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = tid / kMarchGroup;
    const int g = (int)(tid % kMarchGroup);
    if (i >= n) return;
    const float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    const float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    const int j = march_group_bg<kMarchGroup>(b, o, d, t_near[i], t_far[i], grid, nullptr, nullptr,
                                              nullptr, (int32_t)i, g, lane_id() - g);
    if (g == 0) counts[i] = j;
}

__global__ void __launch_bounds__(64) k_march_bg_fill(MarchBgArgs b, const float* __restrict__ rays,
                                                     int64_t n, const float* __restrict__ t_near,
                                                     const float* __restrict__ t_far,
                                                     const uint8_t* __restrict__ grid,
                                                     const int32_t* __restrict__ packed,
                                                     int32_t* __restrict__ ridx,
                                                     float* __restrict__ ts,
                                                     float* __restrict__ te) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = tid / kMarchGroup;
    const int g = (int)(tid % kMarchGroup);
    if (i >= n) return;
    const int32_t base = packed[2 * i];
    const float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    const float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    MarchBgArgs c = b;
    c.m.cap = packed[2 * i + 1];  // never write past the counted samples
    if (c.m.cap == 0) return;
    march_group_bg<kMarchGroup>(c, o, d, t_near[i], t_far[i], grid, ts + base, te + base,
                                ridx + base, (int32_t)i, g, lane_id() - g);
}

// Early-stop visibility of the background samples (nerfacc 0.3.3
// ray_marching with a sigma_fn, alpha_thre 0, as models/neus.py:157-167
// calls it): alpha = 1 - exp(-sigma (t1 - t0)), T_j = prod_{i<j} (1 - alpha_i)
// in sample order, a sample kept while T_j >= eps.  T never grows along a
// ray, so the kept samples are a prefix of the ray's; one lane per ray walks
// it sequentially (the product's rounding order is the sample order).
__global__ void k_visible_prefix(const float* __restrict__ sigma, const float* __restrict__ ts,
                                 const float* __restrict__ te, const int32_t* __restrict__ packed,
                                 int64_t n_rays, float eps, int32_t* __restrict__ keep) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n_rays) return;
    const int32_t b = packed[2 * r], c = packed[2 * r + 1];
    float T = 1.0f;
    int32_t k = 0;
    for (; k < c; ++k) {
        if (!(T >= eps)) break;
        const float alpha = 1.0f - expf(-(sigma[b + k] * (te[b + k] - ts[b + k])));
        T = T * (1.0f - alpha);
    }
    keep[r] = k;
}

__device__ __forceinline__ float ray_near(const float* t_near, const float* jitter, int64_t i,
                                          float step) {
    float nr = t_near[i];
    if (jitter) nr = nr + jitter[i] * step;
    return nr;
}

__global__ void k_ray_aabb(const float* __restrict__ rays, int64_t n, float aabb0, float aabb1,
                           float aabb2, float aabb3, float aabb4, float aabb5,
                           float* __restrict__ t_near, float* __restrict__ t_far) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float aabb[6] = {aabb0, aabb1, aabb2, aabb3, aabb4, aabb5};
    float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    aabb_one(o, d, aabb, t_near + i, t_far + i);
}

template <bool GROUP>
__global__ void __launch_bounds__(256) k_march_count(MarchArgs a, const float* __restrict__ rays,
                                                   int64_t n, const float* __restrict__ t_near,
                                                   const float* __restrict__ t_far,
                                                   const float* __restrict__ jitter,
                                                   const uint8_t* __restrict__ grid,
                                                   int32_t* __restrict__ counts) {
    const int64_t i = march_ray<GROUP>();
    if (i >= n) return;
    const float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    const float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    const int j = march<GROUP>(a, o, d, ray_near(t_near, jitter, i, a.step), t_far[i], grid, nullptr,
                             nullptr, nullptr, (int32_t)i);
    if (march_lead<GROUP>()) counts[i] = j;
}

// packed[i] = (start, count) from counts and their exclusive scan; total.
__global__ void k_march_pack(const int32_t* __restrict__ counts, const int32_t* __restrict__ starts,
                             int64_t n, int32_t* __restrict__ packed, int32_t* __restrict__ total) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n == 0 && i == 0) total[0] = 0;
    if (i >= n) return;
    packed[2 * i] = starts[i];
    packed[2 * i + 1] = counts[i];
    if (i == n - 1) total[0] = starts[i] + counts[i];
}

template <bool GROUP>
__global__ void __launch_bounds__(256) k_march_fill(MarchArgs a, const float* __restrict__ rays,
                                                  int64_t n, const float* __restrict__ t_near,
                                                  const float* __restrict__ t_far,
                                                  const float* __restrict__ jitter,
                                                  const uint8_t* __restrict__ grid,
                                                  const int32_t* __restrict__ packed,
                                                  int32_t* __restrict__ ridx,
                                                  float* __restrict__ ts, float* __restrict__ te) {
    const int64_t i = march_ray<GROUP>();
    if (i >= n) return;
    const int32_t base = packed[2 * i];
    const float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    const float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    MarchArgs b = a;
    b.cap = packed[2 * i + 1];  // never write past the counted samples
    if (b.cap == 0) return;
    march<GROUP>(b, o, d, ray_near(t_near, jitter, i, a.step), t_far[i], grid, ts + base, te + base,
               ridx + base, (int32_t)i);
}

// Staged marching (a per-ray sample cap is set): the count pass also writes
// each ray's samples into a cap-strided staging area, and the fill pass
// copies them to their packed positions instead of marching again.
template <bool GROUP>
__global__ void __launch_bounds__(256) k_march_count_staged(MarchArgs a,
                                                          const float* __restrict__ rays, int64_t n,
                                                          const float* __restrict__ t_near,
                                                          const float* __restrict__ t_far,
                                                          const float* __restrict__ jitter,
                                                          const uint8_t* __restrict__ grid,
                                                          int32_t* __restrict__ counts,
                                                          float* __restrict__ st0,
                                                          float* __restrict__ st1) {
    const int64_t i = march_ray<GROUP>();
    if (i >= n) return;
    const float o[3] = {rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]};
    const float d[3] = {rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]};
    const int64_t base = i * (int64_t)a.cap;   // a.cap > 0: samples j < cap
    const int j = march<GROUP>(a, o, d, ray_near(t_near, jitter, i, a.step), t_far[i], grid,
                             st0 + base, st1 + base, nullptr, (int32_t)i);
    if (march_lead<GROUP>()) counts[i] = j;
}

// One wave per ray: its staged samples to the packed outputs, coalesced.
__global__ void __launch_bounds__(256) k_march_fill_staged(const int32_t* __restrict__ packed,
                                                           int64_t n, int32_t cap,
                                                           const float* __restrict__ st0,
                                                           const float* __restrict__ st1,
                                                           int32_t* __restrict__ ridx,
                                                           float* __restrict__ ts,
                                                           float* __restrict__ te) {
    const int64_t r = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (r >= n) return;
    const int l = threadIdx.x & 63;
    const int32_t base = packed[2 * r], cnt = packed[2 * r + 1];
    const int64_t src = r * (int64_t)cap;
    for (int j = l; j < cnt; j += 64) {
        ts[base + j] = st0[src + j];
        te[base + j] = st1[src + j];
        ridx[base + j] = (int32_t)r;
    }
}

static MarchArgs march_args(const float* roi6, const uint8_t* grid, int res, float step, int cap) {
    MarchArgs a;
    for (int d = 0; d < 6; ++d) a.roi[d] = roi6[d];
    a.res = res;
    a.step = step;
    a.cap = cap;
    a.has_grid = grid != nullptr;
    a.range_pow2 = 0;
    for (int d = 0; d < 3; ++d) {
        const float range = roi6[3 + d] - roi6[d];
        int ex = 0;
        const float m = std::frexp(range, &ex);   // range = m * 2^ex, m in [0.5, 1)
        const bool pow2 = std::isfinite(range) && range > 0.0f && m == 0.5f &&
                          std::isnormal(1.0f / range);
        a.inv_range[d] = pow2 ? 1.0f / range : 0.0f;
        if (pow2) a.range_pow2 |= 1 << d;
    }
    a.res_pow2 = res > 0 && (res & (res - 1)) == 0;
    a.inv_res = a.res_pow2 ? 1.0f / (float)res : 0.0f;
    return a;
}

// Four lanes to a ray or a wave to a ray, once there are enough rays to fill the
// chip either way.  A wave's round costs the same however few of its 64 points
// lie in the box (few steps), or however few cells they cross (cells of many
// steps, which a group skips at once, 16 rays a wave).  Whole call, 128^3 scene
// grid, four lanes against a wave, by steps in the box's diagonal:
//              17         35         49         69         99        1019       3464
//   1048576  324 / 953  503 / 1141 642 / 1203 843 / 1140 1138 / 1314 4384 / 4168 8611 / 11512 us
//    131072   96 / 168  127 / 191  144 / 198  174 / 188  221 / 208   770 / 576   1444 / 1512
//     32768   69 / 82    94 / 91   112 / 91   120 / 93   149 / 98    447 / 212    798 / 455
// (1019 and 3464 steps: 4.6 and 15.6 a cell.)
static bool use_group(const MarchArgs& a, int64_t n_rays) {
    float sq = 0.0f, least = a.roi[3] - a.roi[0];
    for (int d = 0; d < 3; ++d) {
        const float range = a.roi[3 + d] - a.roi[d];
        sq += range * range;
        least = std::fmin(least, range);
    }
    const float steps = std::sqrt(sq) / a.step;
    if (steps <= 80.0f) return (float)n_rays > 1600.0f * steps;
    return a.has_grid && least > 8.0f * (float)a.res * a.step && n_rays > 65536;
}
static unsigned march_blocks(int64_t n_rays, bool group) {
    return (unsigned)ceil_div(n_rays, group ? 256 / kMarchGroup : 4);
}

static size_t scan_tmp_bytes(int64_t n) {
    size_t bytes = 0;
    rocprim::exclusive_scan(nullptr, bytes, (const int32_t*)nullptr, (int32_t*)nullptr, 0,
                            (size_t)n, rocprim::plus<int32_t>(), 0, false);
    return bytes;
}

}  // namespace am

using namespace am;

extern "C" int am_ray_aabb(const float* rays, int64_t n_rays, const float* aabb6_host,
                           float* t_near, float* t_far, void* stream) {
    AM_CHECK_ARG(n_rays >= 0, "n_rays < 0");
    if (n_rays == 0) return AM_OK;
    AM_CHECK_ARG(rays && aabb6_host && t_near && t_far, "NULL buffer");
    const float* b = aabb6_host;
    hipLaunchKernelGGL(k_ray_aabb, dim3((unsigned)ceil_div(n_rays, 256)), dim3(256), 0,
                       to_stream(stream), rays, n_rays, b[0], b[1], b[2], b[3], b[4], b[5], t_near,
                       t_far);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" size_t am_march_workspace_size(int64_t n_rays) {
    if (n_rays < 0) return 0;
    WsCarver c(nullptr, 0);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<char>(scan_tmp_bytes(n_rays > 0 ? n_rays : 1) + 256);
    return c.used + 256;
}

static int check_march(int64_t n_rays, const float* rays, const float* t_near, const float* t_far,
                       const float* roi6, const uint8_t* grid, int32_t res, float step,
                       int32_t cap) {
    AM_CHECK_ARG(n_rays >= 0 && n_rays < (1ll << 31), "n_rays %lld", (long long)n_rays);
    AM_CHECK_ARG(rays && t_near && t_far && roi6, "NULL buffer");
    AM_CHECK_ARG(!grid || (res >= 1 && res <= 4096), "grid_res %d", res);
    AM_CHECK_ARG(step > 0.0f, "step %g <= 0", (double)step);
    AM_CHECK_ARG(cap >= 0, "cap < 0");
    for (int d = 0; d < 3; ++d) AM_CHECK_ARG(roi6[3 + d] > roi6[d], "empty roi");
    return AM_OK;
}

extern "C" int am_march_count(const float* rays, int64_t n_rays, const float* t_near,
                              const float* t_far, const float* jitter, const float* roi6_host,
                              const uint8_t* grid, int32_t grid_res, float step, int32_t cap,
                              int32_t* packed, int32_t* total, void* workspace,
                              size_t workspace_bytes, void* stream) {
    if (int rc = check_march(n_rays, rays, t_near, t_far, roi6_host, grid, grid_res, step, cap))
        return rc;
    AM_CHECK_ARG(packed && total && workspace, "NULL packed/total/workspace");
    hipStream_t s = to_stream(stream);
    if (n_rays == 0) {
        hipLaunchKernelGGL(k_march_pack, dim3(1), dim3(1), 0, s, (const int32_t*)nullptr,
                           (const int32_t*)nullptr, (int64_t)0, packed, total);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    WsCarver c(workspace, workspace_bytes);
    int32_t* counts = c.take<int32_t>((size_t)n_rays + 1);
    int32_t* starts = c.take<int32_t>((size_t)n_rays + 1);
    size_t sb = scan_tmp_bytes(n_rays);
    char* stmp = c.take<char>(sb + 256);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    const MarchArgs a = march_args(roi6_host, grid, grid_res, step, cap);
    const bool group = use_group(a, n_rays);
    {
        KernelTimer kt_("march_count", s);
        auto kern = group ? k_march_count<true> : k_march_count<false>;
        hipLaunchKernelGGL(kern, dim3(march_blocks(n_rays, group)), dim3(256), 0, s, a, rays, n_rays, t_near, t_far,
                           jitter, grid, counts);
    }
    AM_LAUNCH_CHECK();
    hipError_t e = rocprim::exclusive_scan(stmp, sb, counts, starts, 0, (size_t)n_rays,
                                           rocprim::plus<int32_t>(), s, false);
    if (e != hipSuccess) {
        set_error("exclusive scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    hipLaunchKernelGGL(k_march_pack, dim3((unsigned)ceil_div(n_rays, 256)), dim3(256), 0, s, counts,
                       starts, n_rays, packed, total);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_march_fill(const float* rays, int64_t n_rays, const float* t_near,
                             const float* t_far, const float* jitter, const float* roi6_host,
                             const uint8_t* grid, int32_t grid_res, float step, int32_t cap,
                             const int32_t* packed, int32_t* ray_indices, float* t_starts,
                             float* t_ends, void* stream) {
    if (int rc = check_march(n_rays, rays, t_near, t_far, roi6_host, grid, grid_res, step, cap))
        return rc;
    if (n_rays == 0) return AM_OK;
    AM_CHECK_ARG(packed && ray_indices && t_starts && t_ends, "NULL output");
    const MarchArgs a = march_args(roi6_host, grid, grid_res, step, cap);
    {
        KernelTimer kt_("march_fill", to_stream(stream));
        const bool group = use_group(a, n_rays);
        auto kern = group ? k_march_fill<true> : k_march_fill<false>;
        hipLaunchKernelGGL(kern, dim3(march_blocks(n_rays, group)), dim3(256), 0, to_stream(stream), a, rays, n_rays, t_near, t_far, jitter, grid, packed,
                           ray_indices, t_starts, t_ends);
    }
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" size_t am_march_staged_workspace_size(int64_t n_rays, int32_t cap) {
    if (n_rays < 0 || cap <= 0) return 0;
    WsCarver c(nullptr, 0);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<char>(scan_tmp_bytes(n_rays > 0 ? n_rays : 1) + 256);
    c.take<float>((size_t)n_rays * (size_t)cap);
    c.take<float>((size_t)n_rays * (size_t)cap);
    return c.used + 256;
}

extern "C" int am_march_count_staged(const float* rays, int64_t n_rays, const float* t_near,
                                     const float* t_far, const float* jitter,
                                     const float* roi6_host, const uint8_t* grid, int32_t grid_res,
                                     float step, int32_t cap, int32_t* packed, int32_t* total,
                                     void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = check_march(n_rays, rays, t_near, t_far, roi6_host, grid, grid_res, step, cap))
        return rc;
    AM_CHECK_ARG(cap > 0, "staged marching needs a per-ray sample cap (got %d)", cap);
    AM_CHECK_ARG(packed && total && workspace, "NULL packed/total/workspace");
    hipStream_t s = to_stream(stream);
    if (n_rays == 0) {
        hipLaunchKernelGGL(k_march_pack, dim3(1), dim3(1), 0, s, (const int32_t*)nullptr,
                           (const int32_t*)nullptr, (int64_t)0, packed, total);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    WsCarver c(workspace, workspace_bytes);
    int32_t* counts = c.take<int32_t>((size_t)n_rays + 1);
    int32_t* starts = c.take<int32_t>((size_t)n_rays + 1);
    size_t sb = scan_tmp_bytes(n_rays);
    char* stmp = c.take<char>(sb + 256);
    float* st0 = c.take<float>((size_t)n_rays * (size_t)cap);
    float* st1 = c.take<float>((size_t)n_rays * (size_t)cap);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    const MarchArgs a = march_args(roi6_host, grid, grid_res, step, cap);
    {
        KernelTimer kt_("march_count", s);
        const bool group = use_group(a, n_rays);
        auto kern = group ? k_march_count_staged<true> : k_march_count_staged<false>;
        hipLaunchKernelGGL(kern, dim3(march_blocks(n_rays, group)), dim3(256), 0, s, a,
                           rays, n_rays, t_near, t_far, jitter, grid, counts, st0, st1);
    }
    AM_LAUNCH_CHECK();
    hipError_t e = rocprim::exclusive_scan(stmp, sb, counts, starts, 0, (size_t)n_rays,
                                           rocprim::plus<int32_t>(), s, false);
    if (e != hipSuccess) {
        set_error("exclusive scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    hipLaunchKernelGGL(k_march_pack, dim3((unsigned)ceil_div(n_rays, 256)), dim3(256), 0, s, counts,
                       starts, n_rays, packed, total);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_march_fill_staged(int64_t n_rays, int32_t cap, const int32_t* packed,
                                    const void* workspace, size_t workspace_bytes,
                                    int32_t* ray_indices, float* t_starts, float* t_ends,
                                    void* stream) {
    AM_CHECK_ARG(n_rays >= 0 && n_rays < (1ll << 31), "n_rays %lld", (long long)n_rays);
    AM_CHECK_ARG(cap > 0, "staged marching needs a per-ray sample cap (got %d)", cap);
    if (n_rays == 0) return AM_OK;
    AM_CHECK_ARG(packed && workspace && ray_indices && t_starts && t_ends, "NULL buffer");
    // the same carve as am_march_count_staged
    WsCarver c(const_cast<void*>(workspace), workspace_bytes);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<int32_t>((size_t)n_rays + 1);
    c.take<char>(scan_tmp_bytes(n_rays) + 256);
    const float* st0 = c.take<float>((size_t)n_rays * (size_t)cap);
    const float* st1 = c.take<float>((size_t)n_rays * (size_t)cap);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    {
        KernelTimer kt_("march_fill", to_stream(stream));
        hipLaunchKernelGGL(k_march_fill_staged, dim3((unsigned)ceil_div(n_rays, 4)), dim3(256), 0,
                           to_stream(stream), packed, n_rays, cap, st0, st1, ray_indices, t_starts,
                           t_ends);
    }
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_march_bg_count(const float* rays, int64_t n_rays, const float* t_near,
                                 const float* t_far, const float* roi6_host, const uint8_t* grid,
                                 int32_t grid_res, float step, float cone_angle, int32_t cap,
                                 int32_t* packed, int32_t* total, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    if (int rc = check_march(n_rays, rays, t_near, t_far, roi6_host, grid, grid_res, step, cap))
        return rc;
    AM_CHECK_ARG(cone_angle >= 0.0f, "cone_angle %g < 0", (double)cone_angle);
    AM_CHECK_ARG(packed && total && workspace, "NULL output");
    hipStream_t s = to_stream(stream);
    if (n_rays == 0) {
        hipLaunchKernelGGL(k_march_pack, dim3(1), dim3(1), 0, s, (const int32_t*)nullptr,
                           (const int32_t*)nullptr, (int64_t)0, packed, total);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    WsCarver c(workspace, workspace_bytes);
    int32_t* counts = c.take<int32_t>((size_t)n_rays + 1);
    int32_t* starts = c.take<int32_t>((size_t)n_rays + 1);
    size_t sb = scan_tmp_bytes(n_rays);
    char* stmp = c.take<char>(sb + 256);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    MarchBgArgs b;
    b.m = march_args(roi6_host, grid, grid_res, step, cap);
    b.cone = cone_angle;
    {
        KernelTimer kt_("march_bg_count", s);
        hipLaunchKernelGGL(k_march_bg_count, dim3((unsigned)ceil_div(n_rays * kMarchGroup, 64)),
                           dim3(64), 0, s,
                           b, rays, n_rays, t_near, t_far, grid, counts);
    }
    AM_LAUNCH_CHECK();
    hipError_t e = rocprim::exclusive_scan(stmp, sb, counts, starts, 0, (size_t)n_rays,
                                           rocprim::plus<int32_t>(), s, false);
    if (e != hipSuccess) {
        set_error("exclusive scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    hipLaunchKernelGGL(k_march_pack, dim3((unsigned)ceil_div(n_rays, 256)), dim3(256), 0, s, counts,
                       starts, n_rays, packed, total);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_march_bg_fill(const float* rays, int64_t n_rays, const float* t_near,
                                const float* t_far, const float* roi6_host, const uint8_t* grid,
                                int32_t grid_res, float step, float cone_angle, int32_t cap,
                                const int32_t* packed, int32_t* ray_indices, float* t_starts,
                                float* t_ends, void* stream) {
    if (int rc = check_march(n_rays, rays, t_near, t_far, roi6_host, grid, grid_res, step, cap))
        return rc;
    AM_CHECK_ARG(cone_angle >= 0.0f, "cone_angle %g < 0", (double)cone_angle);
    if (n_rays == 0) return AM_OK;
    AM_CHECK_ARG(packed && ray_indices && t_starts && t_ends, "NULL output");
    MarchBgArgs b;
    b.m = march_args(roi6_host, grid, grid_res, step, cap);
    b.cone = cone_angle;
    {
        KernelTimer kt_("march_bg_fill", to_stream(stream));
        hipLaunchKernelGGL(k_march_bg_fill, dim3((unsigned)ceil_div(n_rays * kMarchGroup, 64)),
                           dim3(64), 0,
                           to_stream(stream), b, rays, n_rays, t_near, t_far, grid, packed,
                           ray_indices, t_starts, t_ends);
    }
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_march_bg_visible(const float* sigma, const float* t_starts, const float* t_ends,
                                   const int32_t* packed, int64_t n_rays, float early_stop_eps,
                                   int32_t* packed_out, int32_t* total, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    AM_CHECK_ARG(n_rays >= 0 && n_rays < (1ll << 31), "n_rays %lld", (long long)n_rays);
    AM_CHECK_ARG(packed_out && total, "NULL packed_out/total");
    AM_CHECK_ARG(early_stop_eps >= 0.0f, "early_stop_eps %g < 0", (double)early_stop_eps);
    hipStream_t s = to_stream(stream);
    if (n_rays == 0) {
        hipLaunchKernelGGL(k_march_pack, dim3(1), dim3(1), 0, s, (const int32_t*)nullptr,
                           (const int32_t*)nullptr, (int64_t)0, packed_out, total);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    AM_CHECK_ARG(sigma && t_starts && t_ends && packed && workspace, "NULL buffer");
    WsCarver c(workspace, workspace_bytes);
    int32_t* keep = c.take<int32_t>((size_t)n_rays + 1);
    int32_t* starts = c.take<int32_t>((size_t)n_rays + 1);
    size_t sb = scan_tmp_bytes(n_rays);
    char* stmp = c.take<char>(sb + 256);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    {
        KernelTimer kt_("march_bg_visible", s);
        hipLaunchKernelGGL(k_visible_prefix, dim3((unsigned)ceil_div(n_rays, 64)), dim3(64), 0, s,
                           sigma, t_starts, t_ends, packed, n_rays, early_stop_eps, keep);
    }
    AM_LAUNCH_CHECK();
    hipError_t e = rocprim::exclusive_scan(stmp, sb, keep, starts, 0, (size_t)n_rays,
                                           rocprim::plus<int32_t>(), s, false);
    if (e != hipSuccess) {
        set_error("exclusive scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    hipLaunchKernelGGL(k_march_pack, dim3((unsigned)ceil_div(n_rays, 256)), dim3(256), 0, s, keep,
                       starts, n_rays, packed_out, total);
    AM_LAUNCH_CHECK();
    return AM_OK;
}
