// Arguments and per-sample state of the fused SDF field, shared by its forward
// and backward (geometry.hip) and the table-gradient pair passes (pairs.hip).
#pragma once
#include <type_traits>
#include "hashgrid_dev.h"
#include "mlp_dev.h"
#include "table_grad.h"

namespace am {

struct GeoArgs {
    GridArgs g;
    float r, inv2r, eps, inv_eps, inv_pi;
    int with_grad, with_laplace, recontract, active;
    int n_in, n_out, act;
    float beta;
    int w1, b1, w2, b2, wo, bo, ld1, lds_floats;  // LDS offsets (floats)
    // output tiles of 16 rows (n_out <= 16 * out_tiles); the rows of tiles
    // >= 1 are features only, read by the base evaluation alone
    int out_tiles;
    int64_t pw1, pb1, pw2, pb2, pwo, pbo, n_params;
    int n_evals;  // 1, 7 or 13
    int prec;     // AM_PREC_FP32 / AM_PREC_MIXED
    // analytic-gradient mode: the base evaluation carries d enc / d x and
    // grad = d sdf / d x through the MLP; no FD evaluations.  Slots: curv0 =
    // first curvature evaluation (7 FD mode, 1 analytic), n_dx = stored
    // position-derivative slots (the analytic base, then the 6 curvature
    // evaluations), genc_slots = encode-gradient slots per tile (n_evals, and
    // 3 more in analytic mode: u * scale * g_x along each axis).
    int analytic, curv0, n_dx, dx_curv0, genc_slots;
    // Evaluation order: kernel sample n is the caller's sample order[n]
    // (nullptr: the caller's order).  Inputs (positions, curvature
    // directions, upstream gradients) and outputs are addressed in the
    // caller's order; the forward's saved values (FD values, stored
    // encodings) and the encode gradients in the kernels' order.
    const int32_t* order;
};

__device__ __forceinline__ int64_t caller_row(const GeoArgs& a, int64_t n, bool valid) {
    return (a.order && valid) ? (int64_t)a.order[n] : n;
}
__device__ __forceinline__ float pick3(const float v[3], int k) {
    return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]);
}
__device__ __forceinline__ float contract1(float v, const GeoArgs& a) { return (v + a.r) * a.inv2r; }

__device__ __forceinline__ float clampr(float v, float r) { return fminf(fmaxf(v, -r), r); }

// Offset point j (axis j/2, sign + for even j) around `base` (world units,
// as the reference adds the offsets to it), clamped and contracted; mask =
// the clamp passed the coordinate through.
__device__ __forceinline__ void offset_point(const GeoArgs& a, const float base[3], int j,
                                             float x[3], bool mask[3]) {
    const int ax = j >> 1;
    const float off = (j & 1) ? -a.eps : a.eps;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float v = base[d] + (d == ax ? off : 0.0f);
        mask[d] = v >= -a.r && v <= a.r;
        x[d] = contract1(clampr(v, a.r), a);
    }
}

__device__ __forceinline__ void normalize3(const float v[3], float out[3]) {
    const float n = sqrtf((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    const float d = fmaxf(n, 1e-12f);
#pragma unroll
    for (int q = 0; q < 3; ++q) out[q] = v[q] / d;
}

// Backward of y = v / max(|v|, 1e-12) (F.normalize).
__device__ __forceinline__ void normalize3_bwd(const float v[3], const float g[3], float out[3]) {
    const float n = sqrtf((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    const float d = fmaxf(n, 1e-12f);
    const float gv = g[0] * v[0] + g[1] * v[1] + g[2] * v[2];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        float r = g[q] / d;
        if (n >= 1e-12f) r -= gv / (d * d) * (v[q] / n);
        out[q] = r;
    }
}

__device__ __forceinline__ void cross3(const float a[3], const float b[3], float c[3]) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

// Per-sample state rebuilt from the 12 stored SDF values (all lanes of the
// sample hold it).
struct GeoSample {
    float P[3], x0[3];
    float grad[3], n[3];
    float rn[3], ps[3], grad_s[3], ns[3], dot;
};

__device__ __forceinline__ void diff_pair(float* acc3, int j, float v) {
    // acc[j/2] = f+ then f+ - f- : bit-identical to the single subtraction
    const int ax = j >> 1;
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (d == ax) acc3[d] = (j & 1) ? acc3[d] - v : v;
}

__device__ __forceinline__ void finish_grad(const GeoArgs& a, float g[3]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) g[d] = (0.5f * g[d]) * a.inv_eps;
}

// grad -> normal -> tangent -> shifted point.
__device__ __forceinline__ void geo_tangent(const GeoArgs& a, const float* __restrict__ randn,
                                            int64_t n, bool valid, GeoSample& s) {
    float rd[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) rd[d] = valid ? randn[3 * n + d] : 1.0f;
    normalize3(rd, s.rn);
    float t[3];
    cross3(s.n, s.rn, t);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float base = a.recontract ? s.x0[d] : s.P[d];
        s.ps[d] = base + t[d] * a.eps;
    }
}

// Precision forms of the fused field (template PR).  Mixed: the table rows
// are read in fp16 and the table-gradient pair values are stored in fp16
// (summed in fp32); the SDF MLP stays fp32 in both forms, because the
// central differences of the FD normal divide each evaluation's rounding
// by eps (bf16 activations there gave normals off by 0.3 on average at the
// Neuralangelo shapes, while a fixed fp16 rounding of the table keeps the
// field smooth).
// Table storage of a precision form: fp32 rows, or fp16 rows (mixed form).
template <int PR>
using TableT = typename std::conditional<PR == mlp::kF32, float2, __half2>::type;
// Rebuilds the per-sample state (grad, normal, tangent, curvature terms) of
// the lane's sample from the 12 stored values (6 FD values, or the analytic
// grad in the first 3, then the 6 curvature values).  n: the kernels' index
// (stored values), m: the caller's index (positions, directions).
__device__ __forceinline__ void geo_rebuild(const GeoArgs& a, const float* __restrict__ pts,
                                            const float* __restrict__ randn,
                                            const float* __restrict__ fdv, int64_t n, int64_t m,
                                            bool valid, GeoSample& s) {
#pragma unroll
    for (int d = 0; d < 3; ++d) s.P[d] = valid ? pts[3 * m + d] : 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) s.x0[d] = contract1(s.P[d], a);
    if (a.with_grad) {
        float g[3] = {0.0f, 0.0f, 0.0f};
        if (a.analytic) {
#pragma unroll
            for (int d = 0; d < 3; ++d) g[d] = valid ? fdv[n * 12 + d] : 0.0f;
        } else {
#pragma unroll
            for (int j = 0; j < 6; ++j) diff_pair(g, j, valid ? fdv[n * 12 + j] : 0.0f);
            finish_grad(a, g);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) s.grad[d] = g[d];
        normalize3(s.grad, s.n);
    }
    if (a.with_laplace) {
        geo_tangent(a, randn, m, valid, s);
        float gs[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 6; ++j) diff_pair(gs, j, valid ? fdv[n * 12 + 6 + j] : 0.0f);
        finish_grad(a, gs);
#pragma unroll
        for (int d = 0; d < 3; ++d) s.grad_s[d] = gs[d];
        normalize3(s.grad_s, s.ns);
        s.dot = (s.n[0] * s.ns[0] + s.n[1] * s.ns[1]) + s.n[2] * s.ns[2];
    }
}

// Encode gradients in HBM (written by the backward, read by the pair
// passes): slot 0 base, 1-6 FD, 7-12 curvature (analytic mode: 1-6
// curvature, then three extra slots).  Groups of 64 samples (four tiles):
//   [group][slot][level][feature][64 samples],
// level = lane group + 4 * level slot, so that a wave of the pair passes,
// 64 samples at one level, reads whole rows of 256 bytes and the four tiles
// of a backward block complete them.
__host__ __device__ inline int64_t geo_genc_floats(int64_t tiles, int slots, int LJ) {
    return (tiles + 3) / 4 * slots * LJ * 512;
}
// A lane's first element (level slot 0, feature 0, slot 0) of a tile; slots
// are LJ * 512 floats apart, level slots 512, features 64.
__device__ __forceinline__ int64_t genc_lane(const GeoArgs& a, int64_t tile, int LJ, int lane) {
    return (tile >> 2) * a.genc_slots * (LJ * 512) + (int64_t)((lane >> 4) * 128) +
           (int64_t)((tile & 3) * 16 + (lane & 15));
}

}  // namespace am
