// Fused VolumeSDF.forward (models/geometry.py:195-287) on fp32 MFMA.
//
// One wave evaluates 16 samples.  Per sample: contraction (scale_anything,
// models/utils.py:109-114, with torch's CUDA scalar division = multiply by
// the fp32 reciprocal), the base evaluation, 6 central-difference
// evaluations (:219-234) and, with laplace, 6 around the tangent-shifted
// point (:236-275).  One evaluation = hash-grid encode (lane group k gathers
// levels k, k+4, k+8, k+12 of its sample, which are exactly its MFMA B
// fragments of the first layer) + the SDF MLP on MFMA.  The evaluations run
// in runtime loops so one copy of the encode + MLP body is compiled.
//
// The forward stores the 12 FD / curvature SDF values per sample and, in
// the store form, every evaluation's encoding.  The backward:
//   k_geo_bwd    rebuilds grad, normal, tangent and the curvature terms from
//                the stored values, re-runs each evaluation's MLP forward
//                (from the stored encoding, or a fresh gather in the
//                recompute form), back-propagates it on MFMA and writes the
//                encode gradient to HBM; MLP weight gradients are per-wave
//                register accumulators summed in a fixed order;
//   pairs.hip    turns the encode gradients into table-gradient pairs,
//   table_grad.hip adds them up into dtable.
#include "mlp_dev.h"
#include "pairs.h"
#include "field_common.h"
#include <mutex>

namespace am {
// Row stride (floats) of the 64-column weight matrices in LDS (W2 and the
// output layer): with 67, the row-major reads of the forward (lane i row i,
// lane group k column 4k) and the transposed reads of the backward (lane
// group k row 4k, lane i column i) both hit at most two lanes per bank; 65
// put four on one bank both ways.
constexpr int kWLd = 67;
}  // namespace am

namespace am {

using mlp::krow;

// Row-space column of the SDF MLP first layer for lane-group level slots:
// K-step s < 2LJ -> level k + 4(s/2), feature s%2; s == 2LJ -> xyz[k].
__host__ __device__ inline int geo_col_of_row(int rs, int LJ, int L) {
    const int t = rs >> 4, k = (rs & 15) >> 2, s = 4 * t + (rs & 3);
    if (s < 2 * LJ) {
        const int level = k + 4 * (s >> 1);
        return level < L ? 3 + 2 * level + (s & 1) : -1;
    }
    if (s == 2 * LJ) return k < 3 ? k : -1;
    return -1;
}

template <int LJ>
struct GeoDims {
    static constexpr int KS1 = 2 * LJ + 1;
    static constexpr int IT1 = (KS1 + 3) / 4;
    static constexpr int RS1 = 16 * IT1;
};

template <int LJ, int NH>
__device__ __forceinline__ void geo_load_lds(const GeoArgs& a, const float* __restrict__ params,
                                             float* sm, LevelParams* lv) {
    constexpr int RS1 = GeoDims<LJ>::RS1;
    for (int q = threadIdx.x; q < 64 * RS1; q += blockDim.x) {
        const int o = q / RS1, rs = q - o * RS1;
        const int col = geo_col_of_row(rs, LJ, a.g.L);
        sm[a.w1 + o * a.ld1 + rs] = col >= 0 ? params[a.pw1 + (int64_t)o * a.n_in + col] : 0.0f;
    }
    for (int q = threadIdx.x; q < 64; q += blockDim.x) sm[a.b1 + q] = params[a.pb1 + q];
    if (NH == 2) {
        for (int q = threadIdx.x; q < 64 * 64; q += blockDim.x) {
            const int o = q >> 6, c = q & 63;
            sm[a.w2 + o * kWLd + c] = params[a.pw2 + q];
        }
        for (int q = threadIdx.x; q < 64; q += blockDim.x) sm[a.b2 + q] = params[a.pb2 + q];
    }
    for (int q = threadIdx.x; q < a.out_tiles * 16 * 64; q += blockDim.x) {
        const int o = q >> 6, c = q & 63;
        sm[a.wo + o * kWLd + c] = o < a.n_out ? params[a.pwo + (int64_t)o * 64 + c] : 0.0f;
    }
    for (int q = threadIdx.x; q < a.out_tiles * 16; q += blockDim.x)
        sm[a.bo + q] = q < a.n_out ? params[a.pbo + q] : 0.0f;
    // unrolled: every kernel-argument access has a constant offset (a
    // per-thread index into the by-value struct would copy it to scratch)
#pragma unroll
    for (int q = 0; q < AM_MAX_LEVELS; ++q)
        if ((int)threadIdx.x == q && q < a.g.L) lv[q] = a.g.lv[q];
}

template <int LJ, int NH, bool DX>
struct GeoEval {
    float xb[GeoDims<LJ>::KS1];
    v4f z1[4];
    v4f z2[NH == 2 ? 4 : 1];
    v4f out;
    float dx[DX ? LJ : 1][2][3];
};

// Encode of this lane's level slots at contracted point x (e.xb[0..2LJ),
// and with DX the position derivatives e.dx).
template <int LJ, int NH, bool DX, class TT>
__device__ __forceinline__ void geo_encode(const GeoArgs& a, const LevelParams* lv,
                                           const TT* __restrict__ table, const float x[3],
                                           GeoEval<LJ, NH, DX>& e) {
    const int k = lane_id() >> 4;
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
        const int level = k + 4 * j;
        if (level < a.active) {
            const LevelParams lp = lv[level];
            if constexpr (DX) encode_level_f2<true>(lp, x, table, &e.xb[2 * j], e.dx[j]);
            else encode_level_f2<false>(lp, x, table, &e.xb[2 * j], nullptr);
        } else {
            e.xb[2 * j] = 0.0f;
            e.xb[2 * j + 1] = 0.0f;
            if constexpr (DX) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int d = 0; d < 3; ++d) e.dx[j][f][d] = 0.0f;
            }
        }
    }
}

// ---- offset evaluations from the centre's rows ----
// An evaluation one eps along an axis from its cluster's centre (the base point,
// or the tangent-shifted point) lies in the centre's cell or, mostly, in the
// cell beyond one of its faces: all or half of its 8 rows are the centre's.  So
// the centre's rows of each level slot stay in registers (CentreRows) and an
// evaluation gathers a face's 4 rows, or none; only levels whose cells are
// smaller than eps, and samples outside the box (whose offsets are clamped in
// other axes too), gather more.  Over 16 levels with eps at the finest cell
// that is 17 rows a sample and offset evaluation instead of 128.  The blend is
// the same arithmetic on the same rows.  940 k samples, 16 levels of up to 2^21
// rows, 13 evaluations, with stores: memory reads 13.4 -> 8.3 GB, the kernel
// 3.44 -> 2.80 ms; bound by its two or three waves a SIMD (the rows take 64
// registers) between memory and VALU issue.
template <int LJ, class TT>
struct CentreRows {
    TT v[LJ][8];
};

__device__ __forceinline__ float2 pick(bool c, float2 a, float2 b) {
    return make_float2(c ? a.x : b.x, c ? a.y : b.y);
}
__device__ __forceinline__ __half2 pick(bool c, __half2 a, __half2 b) {
    return __builtin_bit_cast(__half2, c ? __builtin_bit_cast(uint32_t, a)
                                         : __builtin_bit_cast(uint32_t, b));
}

// Whether the centre's rows of this level serve its evaluations.
__device__ __forceinline__ bool near_level(const GeoArgs& a, const LevelParams& lp) {
    return lp.scale * (a.eps * a.inv2r) <= 1.0f;
}

// The centre's rows at contracted point xc: of every active level, or (!ALL)
// of those that serve the evaluations.
template <bool ALL, int LJ, class TT>
__device__ __forceinline__ void centre_rows(const GeoArgs& a, const LevelParams* lv,
                                            const TT* __restrict__ table, const float xc[3],
                                            CentreRows<LJ, TT>& cr) {
    const int k = lane_id() >> 4;
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
        const int level = k + 4 * j;
        if (level < a.active && (ALL || near_level(a, lv[level]))) {
            const LevelParams lp = lv[level];
            const LevelPos p = level_pos(lp, xc);
            uint32_t rows[8];
            cell_rows(lp, p.c, rows);
#pragma unroll
            for (int c = 0; c < 8; ++c) cr.v[j][c] = table[rows[c]];
        }
    }
}

// The centre's own encode from its rows (ALL).
template <int LJ, int NH, bool DX, class TT>
__device__ __forceinline__ void centre_encode(const GeoArgs& a, const LevelParams* lv,
                                              const float xc[3], const CentreRows<LJ, TT>& cr,
                                              GeoEval<LJ, NH, DX>& e) {
    static_assert(!DX, "the base evaluation of the difference form");
    const int k = lane_id() >> 4;
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
        const int level = k + 4 * j;
        e.xb[2 * j] = 0.0f;
        e.xb[2 * j + 1] = 0.0f;
        if (level < a.active) {
            const LevelParams lp = lv[level];
            float2 v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = row2(cr.v[j][c]);
            blend_level_f2<false>(lp, level_pos(lp, xc), v, &e.xb[2 * j], nullptr);
        }
    }
}

// The 4 rows of the face of cell c with the axis coordinate c[AX] + bit, in
// order of the other axes' bits.
template <int AX, class TT>
__device__ __forceinline__ void load_face(const LevelParams& lp, const uint32_t c[3], uint32_t bit,
                                          const TT* __restrict__ table, TT out[4]) {
    const bool hashed = (lp.size_flags & kHashedBit) != 0u;
    const uint32_t m[3] = {1u, hashed ? 2654435761u : lp.res,
                           hashed ? 805459861u : lp.res * lp.res};
    constexpr int b = AX == 0 ? 1 : 0, e = AX == 2 ? 1 : 2;
    const uint32_t cb = c[b] * m[b], ce = c[e] * m[e];
    uint32_t r[4];
    face_rows(lp, (c[AX] + bit) * m[AX], cb, cb + m[b], ce, ce + m[e], r);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = table[lp.offset + r[i]];
}

// Encode at contracted point x, offset along axis AX from the centre xc, two
// slots at a time: both slots' gathers are issued before the first blend, and
// the registers stay within three waves a SIMD.  DX: the position derivatives
// go straight to dx_out (geo_dx layout).
template <int AX, bool DX, int LJ, int NH, class TT>
__device__ __forceinline__ void geo_encode_near(const GeoArgs& a, const LevelParams* lv,
                                                const TT* __restrict__ table, const float xc[3],
                                                const float x[3], const CentreRows<LJ, TT>& cr,
                                                GeoEval<LJ, NH, false>& e,
                                                float* __restrict__ dx_out) {
    constexpr int b = AX == 0 ? 1 : 0, o = AX == 2 ? 1 : 2;
    const int k = lane_id() >> 4;
    const bool line = x[b] == xc[b] && x[o] == xc[o];
#pragma unroll
    for (int h = 0; h < LJ; h += 2) {
        TT face[2][4];   // the high face (up), else the low one
        int dd[2];       // 0, 1, -1: the centre's cell, or beside it; 2: neither
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int level = k + 4 * (h + q);
            dd[q] = 0;
            if (level < a.active) {
                const LevelParams lp = lv[level];
                const LevelPos p = level_pos(lp, x), pc = level_pos(lp, xc);
                const int s = (int)(p.c[AX] - pc.c[AX]);
                dd[q] = line && near_level(a, lp) && s >= -1 && s <= 1 ? s : 2;
                if (dd[q] != 0) load_face<AX>(lp, p.c, dd[q] == 1 ? 1u : 0u, table, face[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int j = h + q, level = k + 4 * j;
            float dx[2][3] = {};
            e.xb[2 * j] = 0.0f;
            e.xb[2 * j + 1] = 0.0f;
            if (level < a.active) {
                const LevelParams lp = lv[level];
                const LevelPos p = level_pos(lp, x);
                float2 v[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int lo = (i & 1) << b | (i >> 1) << o, hi = lo | 1 << AX;
                    const TT cl = cr.v[j][lo], ch = cr.v[j][hi], f = face[q][i];
                    v[lo] = row2(pick(dd[q] == 1, ch, pick(dd[q] == 0, cl, f)));
                    v[hi] = row2(pick(dd[q] == -1, cl, pick(dd[q] == 0, ch, f)));
                }
                if (__builtin_expect(dd[q] == 2, 0)) {   // the high face as well
                    TT high[4];
                    load_face<AX>(lp, p.c, 1u, table, high);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        v[(i & 1) << b | (i >> 1) << o | 1 << AX] = row2(high[i]);
                }
                blend_level_f2<DX>(lp, p, v, &e.xb[2 * j], dx);
            }
            if constexpr (DX) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int d = 0; d < 3; ++d) dx_out[((j * 2 + f) * 3 + d) * 64] = dx[f][d];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Offset evaluation j (0-5) of a cluster.
template <bool DX, int LJ, int NH, class TT>
__device__ __forceinline__ void geo_encode_offset(const GeoArgs& a, const LevelParams* lv,
                                                  const TT* __restrict__ table, const float xc[3],
                                                  const float x[3], int j,
                                                  const CentreRows<LJ, TT>& cr,
                                                  GeoEval<LJ, NH, false>& e,
                                                  float* __restrict__ dx_out) {
    if (j < 2) geo_encode_near<0, DX>(a, lv, table, xc, x, cr, e, dx_out);
    else if (j < 4) geo_encode_near<1, DX>(a, lv, table, xc, x, cr, e, dx_out);
    else geo_encode_near<2, DX>(a, lv, table, xc, x, cr, e, dx_out);
}

// xyz input (last K-step) + SDF MLP forward from the encoded slots up to the
// last hidden pre-activation (all the backward needs).
template <int LJ, int NH, bool DX, int PR>
__device__ __forceinline__ void geo_mlp_hidden(const GeoArgs& a, const float* sm,
                                               const float x[3], GeoEval<LJ, NH, DX>& e) {
    constexpr int KS1 = GeoDims<LJ>::KS1;
    const int k = lane_id() >> 4;
    e.xb[2 * LJ] = k < 3 ? pick3(x, k) * 2.0f - 1.0f : 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) e.z1[t] = mlp::bias_tile(sm + a.b1, t, 64);
    mlp::mm_fwd<KS1, 4, mlp::FragF, PR>(sm + a.w1, a.ld1, mlp::FragF{e.xb}, e.z1);
    if constexpr (NH == 2) {
        v4f h[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) h[t] = mlp::act4(a.act, e.z1[t], a.beta);
#pragma unroll
        for (int t = 0; t < 4; ++t) e.z2[t] = mlp::bias_tile(sm + a.b2, t, 64);
        mlp::mm_fwd<16, 4, mlp::FragV, PR>(sm + a.w2, kWLd, mlp::FragV{h}, e.z2);
    }
}

// The full SDF MLP forward (hidden layers, then the output layer into e.out).
template <int LJ, int NH, bool DX, int PR>
__device__ __forceinline__ void geo_mlp(const GeoArgs& a, const float* sm, const float x[3],
                                        GeoEval<LJ, NH, DX>& e) {
    geo_mlp_hidden<LJ, NH, DX, PR>(a, sm, x, e);
    v4f h[4];
    const v4f* zl = NH == 2 ? e.z2 : e.z1;
#pragma unroll
    for (int t = 0; t < 4; ++t) h[t] = mlp::act4(a.act, zl[t], a.beta);
    e.out = mlp::bias_tile(sm + a.bo, 0, a.n_out);
    mlp::mm_fwd<16, 1, mlp::FragV, PR>(sm + a.wo, kWLd, mlp::FragV{h}, &e.out);
}

// Encode + SDF MLP of this lane's sample at contracted point x.
template <int LJ, int NH, bool DX, int PR, class TT>
__device__ __forceinline__ void geo_eval(const GeoArgs& a, const float* sm,
                                         const LevelParams* lv, const TT* __restrict__ table,
                                         const float x[3], GeoEval<LJ, NH, DX>& e) {
    geo_encode<LJ, NH, DX>(a, lv, table, x, e);
    geo_mlp<LJ, NH, DX, PR>(a, sm, x, e);
}

// Stored encodings (forward -> backward, the "store" form of the backward):
// per tile of 16 samples, evaluation ev (0 base, then 1-6 FD and 7-12
// curvature, or 1-6 curvature in analytic mode) and slot value s < 2LJ, one
// float per lane at
//   enc[((tile * n_evals + ev) * 2LJ + s) * 64 + lane];
// the position derivatives of the evaluations that carry them (dx slot c:
// the analytic base, then the curvature evaluations) follow at
// enc + geo_enc_floats(...):
//   [((tile * n_dx + c) * 6LJ + (j * 2 + f) * 3 + d) * 64 + lane].
// Every access is a 256 B coalesced row.
__host__ __device__ inline int64_t geo_enc_floats(int64_t tiles, int n_evals, int LJ) {
    return tiles * n_evals * 2 * LJ * 64;
}
__host__ __device__ inline int64_t geo_dx_floats(int64_t tiles, int n_dx, int LJ) {
    return tiles * n_dx * 6 * LJ * 64;
}

// This lane's first derivative of dx slot dxs.
__device__ __forceinline__ float* geo_dx_at(float* __restrict__ st, const GeoArgs& a, int64_t tile,
                                            int64_t n_tiles, int dxs, int LJ) {
    return st + geo_enc_floats(n_tiles, a.n_evals, LJ) + (tile * a.n_dx + dxs) * (6 * LJ) * 64 +
           lane_id();
}

template <int LJ, int NH, bool DX>
__device__ __forceinline__ void geo_store(float* __restrict__ st, const GeoArgs& a, int64_t tile,
                                          int64_t n_tiles, int ev, int dxs,
                                          const GeoEval<LJ, NH, DX>& e) {
    const int l = lane_id();
    float* p = st + (tile * a.n_evals + ev) * (2 * LJ) * 64 + l;
#pragma unroll
    for (int q = 0; q < 2 * LJ; ++q) p[q * 64] = e.xb[q];
    if constexpr (DX) {
        float* d0 = geo_dx_at(st, a, tile, n_tiles, dxs, LJ);
#pragma unroll
        for (int j = 0; j < LJ; ++j)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int d = 0; d < 3; ++d) d0[((j * 2 + f) * 3 + d) * 64] = e.dx[j][f][d];
    }
}

template <int LJ, int NH, bool DX>
__device__ __forceinline__ void geo_load(const float* __restrict__ st, const GeoArgs& a,
                                         int64_t tile, int64_t n_tiles, int ev, int dxs,
                                         GeoEval<LJ, NH, DX>& e) {
    const int l = lane_id();
    const float* p = st + (tile * a.n_evals + ev) * (2 * LJ) * 64 + l;
#pragma unroll
    for (int q = 0; q < 2 * LJ; ++q) e.xb[q] = p[q * 64];
    if constexpr (DX) {
        const float* d0 = st + geo_enc_floats(n_tiles, a.n_evals, LJ) +
                          (tile * a.n_dx + dxs) * (6 * LJ) * 64 + l;
#pragma unroll
        for (int j = 0; j < LJ; ++j)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int d = 0; d < 3; ++d) e.dx[j][f][d] = d0[((j * 2 + f) * 3 + d) * 64];
    }
}

// Backward-side evaluation: the stored encoding (ST) or a fresh encode, then
// the MLP forward up to the last hidden pre-activation.
template <int LJ, int NH, bool DX, bool ST, int PR, class TT>
__device__ __forceinline__ void geo_eval_b(const GeoArgs& a, const float* sm, const LevelParams* lv,
                                           const TT* __restrict__ table,
                                           const float* __restrict__ st, int64_t tile,
                                           int64_t n_tiles, int ev, int dxs, const float x[3],
                                           GeoEval<LJ, NH, DX>& e) {
    if constexpr (ST) geo_load<LJ, NH, DX>(st, a, tile, n_tiles, ev, dxs, e);
    else geo_encode<LJ, NH, DX>(a, lv, table, x, e);
    geo_mlp_hidden<LJ, NH, DX, PR>(a, sm, x, e);
}

// sdf and feature outputs of the base evaluation: output tile 0 from e.out,
// the feature rows of tiles >= 1 (n_out > 16) from the last hidden layer.
template <int LJ, int NH, bool DX>
__device__ __forceinline__ void write_base(const GeoArgs& a, const float* sm,
                                           const GeoEval<LJ, NH, DX>& e, const GeoSample& s,
                                           int64_t n, bool valid, int k, int fdim,
                                           float* __restrict__ sdf, float* __restrict__ feature) {
    // (wide outputs come with two hidden layers: make_geo_args rejects them
    // with one, whose kernels keep their registers for the narrow form)
    if (NH == 2 && feature && a.out_tiles > 1) {   // every lane takes part in the MFMA
        v4f h[4];
        const v4f* zl = NH == 2 ? e.z2 : e.z1;
#pragma unroll
        for (int t = 0; t < 4; ++t) h[t] = mlp::act4(a.act, zl[t], a.beta);
#pragma unroll 1
        for (int t = 1; t < a.out_tiles; ++t) {
            v4f o = mlp::bias_tile(sm + a.bo, t, a.n_out);
            mlp::mm_fwd<16, 1, mlp::FragV, mlp::kF32>(sm + a.wo + 16 * t * kWLd, kWLd, mlp::FragV{h},
                                                      &o);
            if (valid)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * t + 4 * k + r;
                    if (row < a.n_out) feature[n * fdim + row] = o[r];
                }
        }
    }
    if (!valid) return;
    if (k == 0) sdf[n] = e.out[0];
    if (feature) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * k + r;
            if (row < a.n_out) feature[n * fdim + row] = e.out[r];
        }
        if (k < 3) feature[n * fdim + a.n_out + k] = pick3(s.x0, k) * 2.0f - 1.0f;
    }
}

// Row 0 of the output layer (the SDF row), Wo[0, hidden], in D-tile layout.
__device__ __forceinline__ void sdf_row_tiles(const GeoArgs& a, const float* sm, v4f w0[4]) {
    const int k = lane_id() >> 4;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) w0[t][r] = sm[a.wo + 16 * t + 4 * k + r];
}

// d sdf / d x01 of the base evaluation (analytic mode): u = W1^T c1, with
// c1 = sigma'(z1) * Wo[0,:] (one hidden layer) or c1 = sigma'(z1) * W2^T
// (sigma'(z2) * Wo[0,:]) (two), is the gradient of the SDF row with respect
// to the MLP input (encoding slots, then xyz*2-1), contracted with the
// encoding's position derivatives e.dx and with 2 for the xyz input; summed
// over the four lane groups (every lane of the sample gets the sum).  u is
// returned in B-fragment layout.
template <int LJ, int NH>
__device__ __forceinline__ void geo_input_grad(const GeoArgs& a, const float* sm,
                                               const GeoEval<LJ, NH, true>& e, float gpos[3],
                                               float u[GeoDims<LJ>::KS1]) {
    constexpr int IT1 = GeoDims<LJ>::IT1;
    const int k = lane_id() >> 4;
    v4f c1[4];
    sdf_row_tiles(a, sm, c1);
    if constexpr (NH == 2) {
        v4f c2[4], e1[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4f h, dh;
            mlp::act_fb4(a.act, e.z2[t], a.beta, h, dh);
            c2[t] = dh * c1[t];
            e1[t] = v4f{0, 0, 0, 0};
        }
        mlp::mm_bwd_in<16, 4, mlp::FragV, mlp::kF32>(sm + a.w2, kWLd, mlp::FragV{c2}, e1);
#pragma unroll
        for (int t = 0; t < 4; ++t) c1[t] = e1[t];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        v4f h, dh;
        mlp::act_fb4(a.act, e.z1[t], a.beta, h, dh);
        c1[t] = dh * c1[t];
    }
    v4f gin[IT1];
#pragma unroll
    for (int t = 0; t < IT1; ++t) gin[t] = v4f{0, 0, 0, 0};
    mlp::mm_bwd_in<16, IT1, mlp::FragV, mlp::kF32>(sm + a.w1, a.ld1, mlp::FragV{c1}, gin);
    const mlp::FragV gb{gin};
#pragma unroll
    for (int q = 0; q < GeoDims<LJ>::KS1; ++q) u[q] = gb[q];
    float gp[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < LJ; ++j)
#pragma unroll
        for (int d = 0; d < 3; ++d) gp[d] += gb[2 * j] * e.dx[j][0][d] + gb[2 * j + 1] * e.dx[j][1][d];
    if (k < 3) {
        const float gxyz = gb[2 * LJ] * 2.0f;
#pragma unroll
        for (int d = 0; d < 3; ++d) gp[d] += d == k ? gxyz : 0.0f;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) gpos[d] = sum_groups(gp[d]);
}

// Forward of the fused field.  AN: analytic-gradient mode (grad from the
// base evaluation's derivatives; one hidden layer), else central
// differences.  fdv keeps, per sample, the 6 FD values (or the analytic
// grad in [0, 3)) and the 6 curvature values, for the backward.
// NEAR: with gradient in the difference form (the offset evaluations run from
// the centre's rows); without it only the base point is evaluated, or, in
// analytic mode, every evaluation gathers its own rows.  Three waves a SIMD
// measured best with NEAR (2.80 ms where two took 2.92 and four, with 123
// registers spilled, 5.6).
template <int LJ, int NH, bool ST, int PR, bool AN, bool NEAR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NEAR ? 3 : 2)))
k_geo_fwd(GeoArgs a, const float* __restrict__ pts,
                                                 const float* __restrict__ randn, int64_t N,
                                                 const void* __restrict__ table_v,
                                                 const float* __restrict__ params,
                                                 float* __restrict__ sdf, float* __restrict__ grad,
                                                 float* __restrict__ normal,
                                                 float* __restrict__ feature,
                                                 float* __restrict__ laplace,
                                                 float* __restrict__ fdv,
                                                 float* __restrict__ store) {
    extern __shared__ float sm[];
    __shared__ LevelParams lv[AM_MAX_LEVELS];
    geo_load_lds<LJ, NH>(a, params, sm, lv);
    __syncthreads();
    const TableT<PR>* table = reinterpret_cast<const TableT<PR>*>(table_v);
    CentreRows<LJ, TableT<PR>> cr;
    const int l = lane_id(), p = l & 15, k = l >> 4;
    const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6;
    const int64_t n_tiles = (N + 15) / 16;
    const int fdim = a.n_out + 3;
    const int vb = xcd_block((int)blockIdx.x, (int)gridDim.x);   // the table gathers share L2
    for (int64_t tile = (int64_t)vb * nw + wave; tile < n_tiles;
         tile += (int64_t)gridDim.x * nw) {
        const int64_t n = tile * 16 + p;
        const bool valid = n < N;
        const int64_t m = caller_row(a, n, valid);
        GeoSample s;
#pragma unroll
        for (int d = 0; d < 3; ++d) s.P[d] = valid ? pts[3 * m + d] : 0.0f;
#pragma unroll
        for (int d = 0; d < 3; ++d) s.x0[d] = contract1(s.P[d], a);
        if constexpr (AN) {
            GeoEval<LJ, NH, true> e;   // with the position derivatives
            geo_eval<LJ, NH, true, mlp::kF32>(a, sm, lv, table, s.x0, e);
            if constexpr (ST) geo_store<LJ, NH, true>(store, a, tile, n_tiles, 0, 0, e);
            write_base(a, sm, e, s, m, valid, k, fdim, sdf, feature);
            if (!a.with_grad) continue;
            float gp[3], u[GeoDims<LJ>::KS1];
            geo_input_grad<LJ, NH>(a, sm, e, gp, u);
#pragma unroll
            for (int d = 0; d < 3; ++d) s.grad[d] = gp[d] * a.inv2r;   // d x01 / d x = 1 / 2r
            if (fdv && valid && k == 0)
#pragma unroll
                for (int d = 0; d < 3; ++d) fdv[n * 12 + d] = s.grad[d];
        } else {
            {
                GeoEval<LJ, NH, false> e;
                if constexpr (NEAR) {
                    centre_rows<true>(a, lv, table, s.x0, cr);
                    centre_encode(a, lv, s.x0, cr, e);
                } else {
                    geo_encode(a, lv, table, s.x0, e);
                }
                if constexpr (ST) geo_store<LJ, NH, false>(store, a, tile, n_tiles, 0, 0, e);
                geo_mlp<LJ, NH, false, mlp::kF32>(a, sm, s.x0, e);
                write_base(a, sm, e, s, m, valid, k, fdim, sdf, feature);
            }
            if constexpr (!NEAR) continue;   // without gradient
            float g[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int j = 0; j < 6; ++j) {
                float x[3];
                bool inb[3];
                offset_point(a, s.P, j, x, inb);
                GeoEval<LJ, NH, false> e;
                geo_encode_offset<false>(a, lv, table, s.x0, x, j, cr, e, nullptr);
                if constexpr (ST) geo_store<LJ, NH, false>(store, a, tile, n_tiles, 1 + j, 0, e);
                geo_mlp<LJ, NH, false, mlp::kF32>(a, sm, x, e);
                const float v = shfl(e.out[0], p);
                diff_pair(g, j, v);
                if (fdv && valid && k == 0) fdv[n * 12 + j] = v;
            }
            finish_grad(a, g);
#pragma unroll
            for (int d = 0; d < 3; ++d) s.grad[d] = g[d];
        }
        normalize3(s.grad, s.n);
        if (valid && k == 0) {
            if (grad)
#pragma unroll
                for (int d = 0; d < 3; ++d) grad[3 * m + d] = s.grad[d];
            if (normal)
#pragma unroll
                for (int d = 0; d < 3; ++d) normal[3 * m + d] = s.n[d];
        }
        if (!a.with_laplace) continue;
        geo_tangent(a, randn, m, valid, s);
        float gs[3] = {0.0f, 0.0f, 0.0f};
        float xc[3];   // the cluster's centre
#pragma unroll
        for (int d = 0; d < 3; ++d) xc[d] = contract1(clampr(s.ps[d], a.r), a);
        if constexpr (NEAR) centre_rows<false>(a, lv, table, xc, cr);
#pragma unroll 1
        for (int j = 0; j < 6; ++j) {
            float x[3];
            bool inb[3];
            offset_point(a, s.ps, j, x, inb);
            float v;
            if constexpr (NEAR) {
                GeoEval<LJ, NH, false> e;
                geo_encode_offset<ST>(a, lv, table, xc, x, j, cr, e,
                                      ST ? geo_dx_at(store, a, tile, n_tiles, a.dx_curv0 + j, LJ)
                                         : nullptr);
                if constexpr (ST)
                    geo_store<LJ, NH, false>(store, a, tile, n_tiles, a.curv0 + j, 0, e);
                geo_mlp<LJ, NH, false, mlp::kF32>(a, sm, x, e);
                v = shfl(e.out[0], p);
            } else {
                GeoEval<LJ, NH, ST> e;  // the store keeps the position derivatives
                geo_eval<LJ, NH, ST, mlp::kF32>(a, sm, lv, table, x, e);
                if constexpr (ST)
                    geo_store<LJ, NH, true>(store, a, tile, n_tiles, a.curv0 + j, a.dx_curv0 + j, e);
                v = shfl(e.out[0], p);
            }
            diff_pair(gs, j, v);
            if (fdv && valid && k == 0) fdv[n * 12 + 6 + j] = v;
        }
        finish_grad(a, gs);
        float ns[3];
        normalize3(gs, ns);
        const float dot = (s.n[0] * ns[0] + s.n[1] * ns[1]) + s.n[2] * ns[2];
        if (valid && k == 0 && laplace) {
            const float lo = -1.0f + 1e-6f, hi = 1.0f - 1e-6f;
            laplace[m] = acosf(fminf(fmaxf(dot, lo), hi)) * a.inv_pi;
        }
    }
}

// ---- backward ----
template <int LJ, int NH>
struct GeoGrad {
    v4f dW1[4 * GeoDims<LJ>::IT1];
    v4f dW2[NH == 2 ? 16 : 1];
    v4f dWo[4];
    v4f db1[4];
    v4f db2[NH == 2 ? 4 : 1];
    v4f dbo;
};

// Feature rows of output tiles >= 1 (n_out > 16) in the base evaluation's
// backward: their upstream gradients come from g_feature, their weight and
// bias gradients accumulate in a wave-private LDS area (acc) instead of
// registers: per tile t >= 1, [4 column tiles][64 lanes] v4f of dWo (the
// mm_dw layout) then 16 row sums of dbo.
struct OutExt {
    const float* g_feature;
    int64_t m;   // the sample's caller row
    int fdim;
    bool valid;
    float* acc;
};
constexpr int kOutExtFloats = 4 * 64 * 4 + 16;   // per extra tile

__device__ __forceinline__ void out_ext_bwd(const GeoArgs& a, const float* sm, const v4f h[4],
                                            const OutExt& x, float* scratch, v4f gh[4]) {
    const int l = lane_id(), i = l & 15, k = l >> 4;
#pragma unroll 1
    for (int t = 1; t < a.out_tiles; ++t) {
        v4f got;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * t + 4 * k + r;
            got[r] = (x.valid && x.g_feature && row < a.n_out) ? x.g_feature[x.m * x.fdim + row]
                                                                 : 0.0f;
        }
        float* acc = x.acc + (t - 1) * kOutExtFloats;
        v4f dw[4];
#pragma unroll
        for (int it = 0; it < 4; ++it) dw[it] = *reinterpret_cast<const v4f*>(acc + (it * 64 + l) * 4);
        mlp::mm_dw<1, 4, 16, mlp::FragV, mlp::kF32>(&got, mlp::FragV{h}, scratch, dw);
#pragma unroll
        for (int it = 0; it < 4; ++it) *reinterpret_cast<v4f*>(acc + (it * 64 + l) * 4) = dw[it];
        const v4f bs = mlp::rowsum_tile(got);
        if (i == 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[1024 + 4 * k + r] += bs[r];
        mlp::mm_bwd_in<4, 4, mlp::FragV, mlp::kF32>(sm + a.wo + 16 * t * kWLd, kWLd, mlp::FragV{&got},
                                                    gh);
    }
}

// LDS float offset of the backward's per-wave OutExt areas (after the
// weights and the four waves' transpose scratch; 16-byte aligned).
__host__ __device__ inline int geo_ext_base(const GeoArgs& a) {
    return (a.lds_floats + 4 * 128 * mlp::kScratchLd + 3) & ~3;
}

// Output-gradient tile with only row 0 (the SDF) set.
__device__ __forceinline__ v4f go_row0(float g) {
    const int k = lane_id() >> 4;
    return v4f{k == 0 ? g : 0.0f, 0.0f, 0.0f, 0.0f};
}

// MLP backward of one evaluation with output gradient `go` (D tile rows =
// outputs): accumulates weight gradients, stores the encode gradient of the
// lane's level slots to genc (the slot's place of genc_lane) and, with DX,
// returns the contracted-position gradient (summed over the 4 lane groups).
template <int LJ, int NH, bool DX, int PR>
__device__ __forceinline__ void geo_eval_bwd(const GeoArgs& a, const float* sm,
                                             const GeoEval<LJ, NH, DX>& e, v4f go,
                                             float* scratch, GeoGrad<LJ, NH>& G, float* genc,
                                             float gpos[3], const OutExt* ext = nullptr) {
    constexpr int KS1 = GeoDims<LJ>::KS1, IT1 = GeoDims<LJ>::IT1;
    const int l = lane_id(), k = l >> 4;
    v4f h[4], dh[4];   // last hidden activation and its derivative
    const v4f* zl = NH == 2 ? e.z2 : e.z1;
#pragma unroll
    for (int t = 0; t < 4; ++t) mlp::act_fb4(a.act, zl[t], a.beta, h[t], dh[t]);
    mlp::mm_dw<1, 4, 16, mlp::FragV, PR>(&go, mlp::FragV{h}, scratch, G.dWo);
    G.dbo += go;
    v4f gh[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) gh[t] = v4f{0, 0, 0, 0};
    mlp::mm_bwd_in<4, 4, mlp::FragV, PR>(sm + a.wo, kWLd, mlp::FragV{&go}, gh);
    if constexpr (NH == 2)
        if (ext) out_ext_bwd(a, sm, h, *ext, scratch, gh);
    if constexpr (NH == 2) {
        v4f gz2[4], h1[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            gz2[t] = gh[t] * dh[t];
            mlp::act_fb4(a.act, e.z1[t], a.beta, h1[t], dh[t]);
            G.db2[t] += gz2[t];
        }
        mlp::mm_dw<4, 4, 16, mlp::FragV, PR>(gz2, mlp::FragV{h1}, scratch, G.dW2);
#pragma unroll
        for (int t = 0; t < 4; ++t) gh[t] = v4f{0, 0, 0, 0};
        mlp::mm_bwd_in<16, 4, mlp::FragV, PR>(sm + a.w2, kWLd, mlp::FragV{gz2}, gh);
    }
    v4f gz1[4];   // dh now holds the first hidden layer's derivative
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        gz1[t] = gh[t] * dh[t];
        G.db1[t] += gz1[t];
    }
    mlp::mm_dw<4, IT1, KS1, mlp::FragF, PR>(gz1, mlp::FragF{e.xb}, scratch, G.dW1);
    v4f gin[IT1];
#pragma unroll
    for (int t = 0; t < IT1; ++t) gin[t] = v4f{0, 0, 0, 0};
    mlp::mm_bwd_in<16, IT1, mlp::FragV, PR>(sm + a.w1, a.ld1, mlp::FragV{gz1}, gin);
    const mlp::FragV gb{gin};  // gb[s] = gradient of B fragment s
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
        genc[j * 512] = gb[2 * j];
        genc[j * 512 + 64] = gb[2 * j + 1];
    }
    if constexpr (DX) {
        float gp[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < LJ; ++j)
#pragma unroll
            for (int d = 0; d < 3; ++d)
                gp[d] += gb[2 * j] * e.dx[j][0][d] + gb[2 * j + 1] * e.dx[j][1][d];
        if (k < 3) {
            const float gxyz = gb[2 * LJ] * 2.0f;
#pragma unroll
            for (int d = 0; d < 3; ++d) gp[d] += d == k ? gxyz : 0.0f;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) gpos[d] = sum_groups(gp[d]);
    }
}

// Backward of the analytic base evaluation.  With v = d input / d x01 . g_x
// (the encoding's position derivatives and 2 for xyz, contracted with the
// upstream gradient of d sdf / d x01), the gradient term of the loss is the
// directional derivative of the SDF row along v: a tangent pass
// s1 = W1 v, a1' = sigma'(z1) s1 (, s2 = W2 a1', a2' = sigma'(z2) s2) and
// sdf' = Wo[0,:] . a_last'.  Its reverse pass, with the ordinary output
// gradient go alongside (adjoints zb of the pre-activations and sb of the
// tangents):
//   dWo += go (x) a_last + e0 (x) a_last'      (e0: row 0 = 1)
//   layer l from the top: sb_l = sigma'(z_l) * ab'_l,
//     zb_l = sigma'(z_l) * ab_l + sigma''(z_l) * s_l * ab'_l,
//     dW_l += zb_l (x) a_{l-1} + sb_l (x) a'_{l-1},  db_l += zb_l,
//     ab_{l-1} = W_l^T zb_l,  ab'_{l-1} = W_l^T sb_l
//   (ab_last = Wo^T go, ab'_last = Wo[0,:]; a_0 = the input, a'_0 = v).
// The input adjoint W1^T zb_1 is the ordinary encode gradient (genc); the
// tangent adjoint u = W1^T sb_1 reaches the table through v: each corner c
// of level l gets u[l,f] * scale_l * grad(w_c) . g_x, stored as
// u[l,f] * scale_l * g_x[d] in three extra slots (gext) for the pair pass.
template <int LJ, int NH>
__device__ __forceinline__ void geo_eval_bwd_an(const GeoArgs& a, const float* sm,
                                                const LevelParams* lv,
                                                const GeoEval<LJ, NH, true>& e, v4f go,
                                                const float gx[3], float* scratch,
                                                GeoGrad<LJ, NH>& G, float* genc, float* gext,
                                                const OutExt* ext) {
    constexpr int KS1 = GeoDims<LJ>::KS1, IT1 = GeoDims<LJ>::IT1;
    const int l = lane_id(), k = l >> 4;
    float v[KS1];
#pragma unroll
    for (int j = 0; j < LJ; ++j)
#pragma unroll
        for (int f = 0; f < 2; ++f)
            v[2 * j + f] = (e.dx[j][f][0] * gx[0] + e.dx[j][f][1] * gx[1]) + e.dx[j][f][2] * gx[2];
    v[2 * LJ] = k < 3 ? 2.0f * pick3(gx, k) : 0.0f;
    v4f h1[4], dh1[4], sv1[4], w0[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        mlp::act_fb4(a.act, e.z1[t], a.beta, h1[t], dh1[t]);
        sv1[t] = v4f{0, 0, 0, 0};
    }
    sdf_row_tiles(a, sm, w0);
    mlp::mm_fwd<KS1, 4, mlp::FragF, mlp::kF32>(sm + a.w1, a.ld1, mlp::FragF{v}, sv1);
    v4f gz1[4], c1[4];   // zb_1 and sb_1
    if constexpr (NH == 1) {
        // output layer: the ordinary term and the gradient term's row 0
        mlp::mm_dw<1, 4, 16, mlp::FragV, mlp::kF32>(&go, mlp::FragV{h1}, scratch, G.dWo);
        G.dbo += go;
        {
            v4f sdh[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) sdh[t] = sv1[t] * dh1[t];
            const v4f e0 = go_row0(1.0f);
            mlp::mm_dw<1, 4, 16, mlp::FragV, mlp::kF32>(&e0, mlp::FragV{sdh}, scratch, G.dWo);
        }
        v4f gh[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) gh[t] = v4f{0, 0, 0, 0};
        mlp::mm_bwd_in<4, 4, mlp::FragV, mlp::kF32>(sm + a.wo, kWLd, mlp::FragV{&go}, gh);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4f d2;
#pragma unroll
            for (int r = 0; r < 4; ++r) d2[r] = mlp::act_d2(a.act, e.z1[t][r], a.beta, dh1[t][r]);
            gz1[t] = gh[t] * dh1[t] + sv1[t] * w0[t] * d2;
            c1[t] = dh1[t] * w0[t];
            G.db1[t] += gz1[t];
        }
    } else {
        // tangent of the second layer
        v4f ad1[4], sv2[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            ad1[t] = dh1[t] * sv1[t];
            sv2[t] = v4f{0, 0, 0, 0};
        }
        mlp::mm_fwd<16, 4, mlp::FragV, mlp::kF32>(sm + a.w2, kWLd, mlp::FragV{ad1}, sv2);
        v4f gz2[4], c2[4];
        {
            v4f h2[4], dh2[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) mlp::act_fb4(a.act, e.z2[t], a.beta, h2[t], dh2[t]);
            mlp::mm_dw<1, 4, 16, mlp::FragV, mlp::kF32>(&go, mlp::FragV{h2}, scratch, G.dWo);
            G.dbo += go;
            {
                v4f ad2[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) ad2[t] = dh2[t] * sv2[t];
                const v4f e0 = go_row0(1.0f);
                mlp::mm_dw<1, 4, 16, mlp::FragV, mlp::kF32>(&e0, mlp::FragV{ad2}, scratch, G.dWo);
            }
            v4f gh[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) gh[t] = v4f{0, 0, 0, 0};
            mlp::mm_bwd_in<4, 4, mlp::FragV, mlp::kF32>(sm + a.wo, kWLd, mlp::FragV{&go}, gh);
            if (ext) out_ext_bwd(a, sm, h2, *ext, scratch, gh);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v4f d2;
#pragma unroll
                for (int r = 0; r < 4; ++r) d2[r] = mlp::act_d2(a.act, e.z2[t][r], a.beta, dh2[t][r]);
                gz2[t] = gh[t] * dh2[t] + sv2[t] * w0[t] * d2;
                c2[t] = dh2[t] * w0[t];
                G.db2[t] += gz2[t];
            }
        }
        mlp::mm_dw<4, 4, 16, mlp::FragV, mlp::kF32>(gz2, mlp::FragV{h1}, scratch, G.dW2);
        mlp::mm_dw<4, 4, 16, mlp::FragV, mlp::kF32>(c2, mlp::FragV{ad1}, scratch, G.dW2);
        v4f gh1[4], e1[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            gh1[t] = v4f{0, 0, 0, 0};
            e1[t] = v4f{0, 0, 0, 0};
        }
        mlp::mm_bwd_in<16, 4, mlp::FragV, mlp::kF32>(sm + a.w2, kWLd, mlp::FragV{gz2}, gh1);
        mlp::mm_bwd_in<16, 4, mlp::FragV, mlp::kF32>(sm + a.w2, kWLd, mlp::FragV{c2}, e1);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4f d2;
#pragma unroll
            for (int r = 0; r < 4; ++r) d2[r] = mlp::act_d2(a.act, e.z1[t][r], a.beta, dh1[t][r]);
            gz1[t] = gh1[t] * dh1[t] + sv1[t] * e1[t] * d2;
            c1[t] = dh1[t] * e1[t];
            G.db1[t] += gz1[t];
        }
    }
    mlp::mm_dw<4, IT1, KS1, mlp::FragF, mlp::kF32>(gz1, mlp::FragF{e.xb}, scratch, G.dW1);
    mlp::mm_dw<4, IT1, KS1, mlp::FragF, mlp::kF32>(c1, mlp::FragF{v}, scratch, G.dW1);
    v4f gin[IT1], uin[IT1];
#pragma unroll
    for (int t = 0; t < IT1; ++t) {
        gin[t] = v4f{0, 0, 0, 0};
        uin[t] = v4f{0, 0, 0, 0};
    }
    mlp::mm_bwd_in<16, IT1, mlp::FragV, mlp::kF32>(sm + a.w1, a.ld1, mlp::FragV{gz1}, gin);
    mlp::mm_bwd_in<16, IT1, mlp::FragV, mlp::kF32>(sm + a.w1, a.ld1, mlp::FragV{c1}, uin);
    const mlp::FragV gb{gin}, ub{uin};
#pragma unroll
    for (int j = 0; j < LJ; ++j) {
        genc[j * 512] = gb[2 * j];
        genc[j * 512 + 64] = gb[2 * j + 1];
        const int level = k + 4 * j;
        const float sc = level < a.g.L ? lv[level].scale : 0.0f;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            gext[d * LJ * 512 + j * 512] = ub[2 * j] * sc * gx[d];
            gext[d * LJ * 512 + j * 512 + 64] = ub[2 * j + 1] * sc * gx[d];
        }
    }
}

template <int LJ, int NH, bool ST, int PR, bool AN>
__device__ __forceinline__ void geo_bwd_body(
    const GeoArgs& a, const float* __restrict__ pts,
    const float* __restrict__ randn, int64_t N, const void* __restrict__ table_v,
    const float* __restrict__ params, const float* __restrict__ fdv,
    const float* __restrict__ store,
    const float* __restrict__ g_sdf, const float* __restrict__ g_grad,
    const float* __restrict__ g_normal, const float* __restrict__ g_feature,
    const float* __restrict__ g_laplace, float* __restrict__ genc_g,
    float* __restrict__ partial) {
    extern __shared__ float sm[];
    __shared__ LevelParams lv[AM_MAX_LEVELS];
    geo_load_lds<LJ, NH>(a, params, sm, lv);
    __syncthreads();
    const TableT<PR>* table = reinterpret_cast<const TableT<PR>*>(table_v);
    const int l = lane_id(), p = l & 15, k = l >> 4;
    const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6;
    float* scratch = sm + a.lds_floats + wave * (128 * mlp::kScratchLd);
    // accumulators of the feature rows of output tiles >= 1 (n_out > 16, two
    // hidden layers)
    const int ext_floats = NH == 2 ? (a.out_tiles - 1) * kOutExtFloats : 0;
    float* ext_acc = sm + geo_ext_base(a) + wave * ext_floats;
    for (int q = l; q < ext_floats; q += 64) ext_acc[q] = 0.0f;
    mlp::wave_sync();
    const int64_t n_tiles = (N + 15) / 16;
    const int fdim = a.n_out + 3;
    GeoGrad<LJ, NH> G;
#pragma unroll
    for (int q = 0; q < 4 * GeoDims<LJ>::IT1; ++q) G.dW1[q] = v4f{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < (NH == 2 ? 16 : 1); ++q) G.dW2[q] = v4f{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        G.dWo[q] = v4f{0, 0, 0, 0};
        G.db1[q] = v4f{0, 0, 0, 0};
    }
#pragma unroll
    for (int q = 0; q < (NH == 2 ? 4 : 1); ++q) G.db2[q] = v4f{0, 0, 0, 0};
    G.dbo = v4f{0, 0, 0, 0};

    for (int64_t tile = (int64_t)blockIdx.x * nw + wave; tile < n_tiles;
         tile += (int64_t)gridDim.x * nw) {
        const int64_t n = tile * 16 + p;
        const bool valid = n < N;
        const int64_t m = caller_row(a, n, valid);
        // this tile's encode-gradient slots (0 base, then FD and curvature, or
        // curvature and the three analytic extra slots)
        float* genc = genc_g + genc_lane(a, tile, LJ, l);
        GeoSample s;
        geo_rebuild(a, pts, randn, fdv, n, m, valid, s);
        // upstream gradients of this sample
        float gg[3] = {0, 0, 0}, gnrm[3] = {0, 0, 0};
        if (valid && g_grad)
#pragma unroll
            for (int d = 0; d < 3; ++d) gg[d] = g_grad[3 * m + d];
        if (valid && g_normal)
#pragma unroll
            for (int d = 0; d < 3; ++d) gnrm[d] = g_normal[3 * m + d];
        // output gradient of the base evaluation
        v4f go;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * k + r;
            float v = 0.0f;
            if (valid && row < a.n_out) {
                if (g_feature) v = g_feature[m * fdim + row];
                if (row == 0 && g_sdf) v += g_sdf[m];
            }
            go[r] = v;
        }
        if constexpr (!AN) {   // base evaluation (genc slot 0)
            GeoEval<LJ, NH, false> e;
            geo_eval_b<LJ, NH, false, ST, mlp::kF32>(a, sm, lv, table, store, tile, n_tiles, 0, 0,
                                                     s.x0, e);
            const OutExt ext{g_feature, m, fdim, valid, ext_acc};
            geo_eval_bwd<LJ, NH, false, mlp::kF32>(a, sm, e, go, scratch, G, genc, nullptr,
                                                   a.out_tiles > 1 ? &ext : nullptr);
        }
        if (a.with_laplace) {
            const float gl = (valid && g_laplace) ? g_laplace[m] : 0.0f;
            const float lo = -1.0f + 1e-6f, hi = 1.0f - 1e-6f;
            const float dc = fminf(fmaxf(s.dot, lo), hi);
            const bool pass = s.dot >= lo && s.dot <= hi;
            const float g_dot = pass ? (gl * a.inv_pi) * (-1.0f / sqrtf(1.0f - dc * dc)) : 0.0f;
            float g_ns[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                gnrm[d] += g_dot * s.ns[d];
                g_ns[d] = g_dot * s.n[d];
            }
            float g_gs[3];
            normalize3_bwd(s.grad_s, g_ns, g_gs);
            float g_ps[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int j = 0; j < 6; ++j) {
                const float ggs = pick3(g_gs, j >> 1);
                const float gf = (j & 1 ? -0.5f : 0.5f) * a.inv_eps * ggs;
                float x[3];
                bool inb[3];
                offset_point(a, s.ps, j, x, inb);
                GeoEval<LJ, NH, true> e;
                geo_eval_b<LJ, NH, true, ST, mlp::kF32>(a, sm, lv, table, store, tile, n_tiles,
                                                        a.curv0 + j, a.dx_curv0 + j, x, e);
                float gpos[3];
                geo_eval_bwd<LJ, NH, true, mlp::kF32>(a, sm, e, go_row0(gf), scratch, G,
                                                      genc + (a.curv0 + j) * LJ * 512, gpos);
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (inb[d]) g_ps[d] += gpos[d] * a.inv2r;
            }
            float g_t[3], gcr[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) g_t[d] = g_ps[d] * a.eps;
            cross3(s.rn, g_t, gcr);
#pragma unroll
            for (int d = 0; d < 3; ++d) gnrm[d] += gcr[d];
        }
        if constexpr (AN) {
            // analytic mode: the base evaluation with the second-order terms
            // of the gradient output (with_grad holds in this mode)
            float gn2g[3];
            normalize3_bwd(s.grad, gnrm, gn2g);
            float gx[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) gx[d] = (gg[d] + gn2g[d]) * a.inv2r;
            GeoEval<LJ, NH, true> e;
            geo_eval_b<LJ, NH, true, ST, mlp::kF32>(a, sm, lv, table, store, tile, n_tiles, 0, 0,
                                                    s.x0, e);
            const OutExt ext{g_feature, m, fdim, valid, ext_acc};
            geo_eval_bwd_an<LJ, NH>(a, sm, lv, e, go, gx, scratch, G, genc,
                                    genc + a.n_evals * LJ * 512, a.out_tiles > 1 ? &ext : nullptr);
        } else if (a.with_grad) {
            float gn2g[3];
            normalize3_bwd(s.grad, gnrm, gn2g);
#pragma unroll
            for (int d = 0; d < 3; ++d) gg[d] += gn2g[d];
#pragma unroll 1
            for (int j = 0; j < 6; ++j) {
                const float gf = (j & 1 ? -0.5f : 0.5f) * a.inv_eps * pick3(gg, j >> 1);
                float x[3];
                bool inb[3];
                offset_point(a, s.P, j, x, inb);
                GeoEval<LJ, NH, false> e;
                geo_eval_b<LJ, NH, false, ST, mlp::kF32>(a, sm, lv, table, store, tile, n_tiles,
                                                         1 + j, 0, x, e);
                geo_eval_bwd<LJ, NH, false, mlp::kF32>(a, sm, e, go_row0(gf), scratch, G,
                                                       genc + (1 + j) * LJ * 512, nullptr);
            }
        }
    }
    // per-wave partial gradient row in parameter layout
    float* out = partial + ((int64_t)blockIdx.x * nw + wave) * a.n_params;
    const int i = p;
    constexpr int IT1 = GeoDims<LJ>::IT1;
#pragma unroll
    for (int ot = 0; ot < 4; ++ot)
#pragma unroll
        for (int it = 0; it < IT1; ++it)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 16 * ot + 4 * k + r;
                const int col = geo_col_of_row(16 * it + i, LJ, a.g.L);
                if (col >= 0) out[a.pw1 + (int64_t)o * a.n_in + col] = G.dW1[ot * IT1 + it][r];
            }
    if constexpr (NH == 2) {
#pragma unroll
        for (int ot = 0; ot < 4; ++ot)
#pragma unroll
            for (int it = 0; it < 4; ++it)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[a.pw2 + (16 * ot + 4 * k + r) * 64 + 16 * it + i] = G.dW2[ot * 4 + it][r];
    }
#pragma unroll
    for (int it = 0; it < 4; ++it)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 4 * k + r;
            if (o < a.n_out) out[a.pwo + o * 64 + 16 * it + i] = G.dWo[it][r];
        }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const v4f s1 = mlp::rowsum_tile(G.db1[t]);
        if (i == 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[a.pb1 + 16 * t + 4 * k + r] = s1[r];
        if constexpr (NH == 2) {
            const v4f s2 = mlp::rowsum_tile(G.db2[t]);
            if (i == 0)
#pragma unroll
                for (int r = 0; r < 4; ++r) out[a.pb2 + 16 * t + 4 * k + r] = s2[r];
        }
    }
    const v4f so = mlp::rowsum_tile(G.dbo);
    if (i == 0)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * k + r < a.n_out) out[a.pbo + 4 * k + r] = so[r];
    // feature rows of output tiles >= 1
    mlp::wave_sync();
#pragma unroll 1
    for (int t = 1; t < (NH == 2 ? a.out_tiles : 1); ++t) {
        const float* acc = ext_acc + (t - 1) * kOutExtFloats;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const v4f dw = *reinterpret_cast<const v4f*>(acc + (it * 64 + l) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 16 * t + 4 * k + r;
                if (o < a.n_out) out[a.pwo + o * 64 + 16 * it + i] = dw[r];
            }
        }
        if (i == 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = 16 * t + 4 * k + r;
                if (o < a.n_out) out[a.pbo + o] = acc[1024 + 4 * k + r];
            }
    }
}

#define AM_GEO_BWD_PARAMS                                                                  \
    GeoArgs a, const float* __restrict__ pts, const float* __restrict__ randn, int64_t N,      \
        const void* __restrict__ table_v, const float* __restrict__ params,                    \
        const float* __restrict__ fdv, const float* __restrict__ store,                        \
        const float* __restrict__ g_sdf, const float* __restrict__ g_grad,                     \
        const float* __restrict__ g_normal, const float* __restrict__ g_feature,               \
        const float* __restrict__ g_laplace, float* __restrict__ genc_g,                       \
        float* __restrict__ partial
#define AM_GEO_BWD_ARGS                                                                     \
    a, pts, randn, N, table_v, params, fdv, store, g_sdf, g_grad, g_normal, g_feature,          \
        g_laplace, genc_g, partial

template <int LJ, int NH, bool ST, int PR, bool AN>
__global__ void __launch_bounds__(256) k_geo_bwd(AM_GEO_BWD_PARAMS) {
    geo_bwd_body<LJ, NH, ST, PR, AN>(AM_GEO_BWD_ARGS);
}

// The 1-hidden-layer form at two waves per SIMD: its state fits the 256
// registers a lane has at that occupancy with a small spill, and the second
// wave hides the LDS and memory latency of the first.
template <int LJ, bool ST, int PR, bool AN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_geo_bwd_o2(AM_GEO_BWD_PARAMS) {
    geo_bwd_body<LJ, 1, ST, PR, AN>(AM_GEO_BWD_ARGS);
}

// ------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------
static int make_geo_args(const am_grid_desc* g, const am_mlp_desc* m, const am_sdf_desc* s,
                         GeoArgs* out, int* LJ) {
    AM_CHECK_ARG(g && m && s, "NULL descriptor");
    if (int rc = check_mlp_common(m, kGeoMaxOut)) return rc;
    if (m->n_out > 16 && m->n_hidden_layers != 2) {
        set_error("an SDF MLP with more than 16 outputs (got %d) takes two hidden layers",
                  m->n_out);
        return AM_ERR_UNSUPPORTED;
    }
    AM_CHECK_ARG(g->n_features == 2, "fused geometry needs n_features = 2 (got %d)", g->n_features);
    AM_CHECK_ARG(g->n_levels >= 1 && g->n_levels <= 16, "fused geometry needs <= 16 levels");
    AM_CHECK_ARG(m->n_in == 3 + 2 * g->n_levels, "SDF MLP n_in %d != 3 + L*F", m->n_in);
    AM_CHECK_ARG(s->active_levels >= 0 && s->active_levels <= g->n_levels, "active_levels %d",
                 s->active_levels);
    AM_CHECK_ARG(s->radius > 0.0f, "radius <= 0");
    AM_CHECK_ARG(s->grad_type == AM_GRAD_FD || s->grad_type == AM_GRAD_ANALYTIC, "grad_type %d",
                 s->grad_type);
    const bool analytic = s->with_grad && s->grad_type == AM_GRAD_ANALYTIC;
    AM_CHECK_ARG(!(s->with_laplace || (s->with_grad && !analytic)) || s->fd_eps > 0.0f,
                 "fd_eps <= 0");
    AM_CHECK_ARG(!s->with_laplace || s->with_grad, "laplace needs with_grad");
    AM_CHECK_ARG(s->precision == AM_PREC_FP32 || s->precision == AM_PREC_MIXED,
                 "precision %d", s->precision);
    AM_CHECK_ARG(m->precision == AM_PREC_FP32,
                 "the SDF MLP runs in fp32 in every form (got precision %d): central "
                 "differences amplify per-evaluation rounding by 1/eps", m->precision);
    GeoArgs a{};
    a.g = make_grid_args(g);
    a.r = s->radius;
    a.inv2r = 1.0f / (float)(2.0 * (double)s->radius);
    a.eps = s->fd_eps;
    a.inv_eps = 1.0f / s->fd_eps;
    a.inv_pi = 1.0f / (float)M_PI;
    a.with_grad = s->with_grad;
    a.with_laplace = s->with_laplace;
    a.recontract = s->recontract;
    a.active = s->active_levels;
    a.n_in = m->n_in;
    a.n_out = m->n_out;
    a.act = m->hidden_act;
    a.beta = m->softplus_beta;
    // level slots per lane group: 2 (L <= 8) or 4 (L <= 16); spare slots
    // hold levels >= L and stay zero.
    const int lj = g->n_levels <= 8 ? 2 : 4;
    const int rs1 = 16 * ((2 * lj + 1 + 3) / 4);
    a.ld1 = rs1 + 1;
    int o = 0;
    a.w1 = o; o += 64 * a.ld1;
    a.b1 = o; o += 64;
    a.w2 = o; a.b2 = o;
    if (m->n_hidden_layers == 2) { a.w2 = o; o += 64 * kWLd; a.b2 = o; o += 64; }
    a.out_tiles = (m->n_out + 15) / 16;
    a.wo = o; o += a.out_tiles * 16 * kWLd;
    a.bo = o; o += a.out_tiles * 16;
    a.lds_floats = o;
    layout_params(m->n_in, m->n_out, m->n_hidden_layers, &a.pw1, &a.pb1, &a.pw2, &a.pb2, &a.pwo,
                  &a.pbo, &a.n_params);
    a.analytic = analytic ? 1 : 0;
    a.n_evals = 1 + (s->with_grad && !analytic ? 6 : 0) + (s->with_laplace ? 6 : 0);
    a.curv0 = analytic ? 1 : 7;
    a.dx_curv0 = analytic ? 1 : 0;
    a.n_dx = (analytic ? 1 : 0) + (s->with_laplace ? 6 : 0);
    a.genc_slots = a.n_evals + (analytic ? 3 : 0);
    a.prec = s->precision;
    *out = a;
    *LJ = lj;
    return AM_OK;
}

template <int LJ, int NH, bool ST, int PR>
static int geo_fwd_launch_t(const GeoArgs& a, const float* pts, const float* randn, int64_t n,
                            const void* table, const float* params, float* sdf, float* grad,
                            float* normal, float* feature, float* laplace, float* fdv,
                            float* store, hipStream_t s) {
    const size_t lds = (size_t)a.lds_floats * sizeof(float);
    auto kern = a.analytic    ? k_geo_fwd<LJ, NH, ST, PR, true, false>
                : a.with_grad ? k_geo_fwd<LJ, NH, ST, PR, false, true>
                              : k_geo_fwd<LJ, NH, ST, PR, false, false>;
    AM_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
    {
        KernelTimer kt_("geo_fwd", s);
        const int most = a.analytic ? kFwdBlocksAnalytic
                                    : (a.with_grad ? kFwdBlocksNear : kFwdBlocksBase);
        const int nb = persistent_blocks((n + 15) / 16, 4, most);
        hipLaunchKernelGGL(kern, dim3(nb), dim3(256), lds, s, a, pts, randn, n, table, params, sdf, grad, normal, feature, laplace, fdv, store);
    }
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <int LJ, int NH>
static int geo_fwd_launch(const GeoArgs& a, const float* pts, const float* randn, int64_t n,
                          const void* table, const float* params, float* sdf, float* grad,
                          float* normal, float* feature, float* laplace, float* fdv, float* store,
                          hipStream_t s) {
    if (a.prec == AM_PREC_MIXED) {
        if (store)
            return geo_fwd_launch_t<LJ, NH, true, mlp::kBF16>(a, pts, randn, n, table, params, sdf,
                                                              grad, normal, feature, laplace, fdv,
                                                              store, s);
        return geo_fwd_launch_t<LJ, NH, false, mlp::kBF16>(a, pts, randn, n, table, params, sdf,
                                                           grad, normal, feature, laplace, fdv,
                                                           nullptr, s);
    }
    if (store)
        return geo_fwd_launch_t<LJ, NH, true, mlp::kF32>(a, pts, randn, n, table, params, sdf,
                                                         grad, normal, feature, laplace, fdv,
                                                         store, s);
    return geo_fwd_launch_t<LJ, NH, false, mlp::kF32>(a, pts, randn, n, table, params, sdf, grad,
                                                      normal, feature, laplace, fdv, nullptr, s);
}

// The backward's workspace before the pair arrays: the pair count is only
// known after the count pass, so the pair arrays are carved afterwards
// from the rest (sized for the worst case by the size query).
struct GeoBwdWs {
    float* fdv;
    float* sdf_tmp;
    float* genc;
    float* partial;
    float* ctmp;
    PairHead pairs;
};

static void carve_geo_bwd_head(WsCarver& c, const GeoArgs& a, const am_grid_desc* g, int LJ,
                               int64_t n, bool need_fdv, GeoBwdWs* w) {
    const int waves = bwd_blocks(n) * 4;
    const int64_t tiles = (n + 15) / 16;
    w->fdv = need_fdv ? c.take<float>((size_t)n * 12 + 1) : nullptr;
    w->sdf_tmp = need_fdv ? c.take<float>((size_t)n + 1) : nullptr;
    w->genc = c.take<float>((size_t)geo_genc_floats(tiles, a.genc_slots, LJ) + 1);
    w->partial = c.take<float>((size_t)waves * a.n_params);
    w->ctmp = c.take<float>((size_t)colsum_tmp_floats(waves, a.n_params) + 1);
    pairs_carve(c, a, g, n, &w->pairs);
}

// The pair arrays for a count pass's capacity (pages, or pairs).
static int carve_pairs(WsCarver& c, const GeoArgs& a, const am_grid_desc* g, const PairHead& h,
                       int64_t capacity, TablePages* tp, TableReduceWs* tw) {
    const bool half = a.prec == AM_PREC_MIXED;
    if (!h.paged) return table_reduce_carve(c, g, capacity, tw, half);
    const int64_t cut = flag_value("sdf_bwd_page_cut", 0);   // (tests)
    if (cut > 0) capacity = capacity > cut ? capacity - cut : 0;
    table_pages_carve(c, g, capacity, half, tp);
    return AM_OK;
}

// Consistency flags of recent backward calls.  The emission flags a page
// (sorted form: a tile) whose pairs are not as many as the count pass found;
// instead of a stream sync per call, each call copies its flag into a pinned
// host slot behind an event, and later calls (after their own pair-count sync,
// cheaply) and am_sdf_bwd_check read the slots whose copies have landed.  A
// mismatch gives a wrong dtable, never a stray access: pairs stay inside their
// page, which holds only pairs put and counted, every page that the reduction
// walks has its run table and lies inside the arrays, and rows are taken modulo
// the bucket (sorted form: pairs stay inside their tile's reserved range, and
// the sort and reduce only index rows below n_entries and items below the
// count whatever the keys hold).
namespace {
struct FlagSlot {
    hipEvent_t ev = nullptr;
    int64_t* flag = nullptr;   // pinned host memory
    bool armed = false;
};
constexpr int kFlagSlots = 16;
std::mutex g_flag_mu;
FlagSlot g_flag_slots[kFlagSlots];
int g_flag_next = 0;
}  // namespace

static int flag_result(FlagSlot& f) {
    f.armed = false;
    if (*f.flag != 0) {
        set_error("table-gradient pair count mismatch between the count and emit passes of an "
                  "earlier am_sdf_bwd call");
        return AM_ERR_INTERNAL;
    }
    return AM_OK;
}

// Reads the armed slots: those whose copy has landed, or all (wait).
static int collect_flags(bool wait) {
    std::lock_guard<std::mutex> lk(g_flag_mu);
    int rc = AM_OK;
    for (FlagSlot& f : g_flag_slots) {
        if (!f.armed) continue;
        const hipError_t e = wait ? hipEventSynchronize(f.ev) : hipEventQuery(f.ev);
        if (e == hipErrorNotReady) continue;
        if (e != hipSuccess) {
            set_error("consistency flag event failed: %s", hipGetErrorString(e));
            return AM_ERR_HIP;
        }
        if (int r = flag_result(f)) rc = r;
    }
    return rc;
}

static int arm_flag(const int64_t* dev_flag, hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_flag_mu);
    FlagSlot& f = g_flag_slots[g_flag_next];
    g_flag_next = (g_flag_next + 1) % kFlagSlots;
    if (f.ev == nullptr) {
        AM_HIP(hipEventCreateWithFlags(&f.ev, hipEventDisableTiming));
        AM_HIP(hipHostMalloc((void**)&f.flag, sizeof(int64_t), hipHostMallocDefault));
    } else if (f.armed) {   // the ring wrapped onto a pending slot
        AM_HIP(hipEventSynchronize(f.ev));
        if (int rc = flag_result(f)) return rc;
    }
    AM_HIP(hipMemcpyAsync(f.flag, dev_flag, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    AM_HIP(hipEventRecord(f.ev, s));
    f.armed = true;
    return AM_OK;
}

template <int LJ, int NH, int PR>
static int geo_bwd_launch_t(const GeoArgs& a, const am_grid_desc* g, const float* pts,
                            const float* randn, int64_t n, const void* table, const float* params,
                            const float* fdv_in,
                          const float* store, const float* g_sdf, const float* g_grad,
                          const float* g_normal, const float* g_feature, const float* g_laplace,
                          float* dtable, float* dparams, void* ws, size_t ws_bytes, hipStream_t s) {
    const int blocks = bwd_blocks(n);
    const int waves = blocks * 4;
    const int64_t tiles = (n + 15) / 16;
    const bool need_fdv = a.with_grad && fdv_in == nullptr;
    AM_CHECK_ARG(!store || !need_fdv, "a stored encoding needs the stored FD values too");
    WsCarver c(ws, ws_bytes);
    GeoBwdWs w;
    carve_geo_bwd_head(c, a, g, LJ, n, need_fdv, &w);
    if (!c.ok()) return workspace_short(c.used, ws_bytes);
    const float* fdv = fdv_in;
    if (need_fdv) {  // recompute the stored SDF values with a forward pass
        if (int rc = geo_fwd_launch<LJ, NH>(a, pts, randn, n, table, params, w.sdf_tmp, nullptr,
                                            nullptr, nullptr, nullptr, w.fdv, nullptr, s))
            return rc;
        fdv = w.fdv;
    }
    // the backward proper: MLP parameter partials and the encode gradients
    auto launch_bwd = [&]() -> int {
        const size_t lds =
            (size_t)(geo_ext_base(a) + 4 * (a.out_tiles - 1) * kOutExtFloats) * sizeof(float);
        AM_CHECK_ARG(lds <= 160 * 1024, "geometry backward needs %zu bytes of LDS", lds);
        auto kern = k_geo_bwd_o2<LJ, true, PR, false>;   // the type of every form's kernel
        if constexpr (NH == 1) {
            kern = store ? k_geo_bwd_o2<LJ, true, PR, false> : k_geo_bwd_o2<LJ, false, PR, false>;
            if (a.analytic)
                kern = store ? k_geo_bwd_o2<LJ, true, PR, true> : k_geo_bwd_o2<LJ, false, PR, true>;
        } else {
            kern = store ? k_geo_bwd<LJ, NH, true, PR, false> : k_geo_bwd<LJ, NH, false, PR, false>;
            if (a.analytic)
                kern = store ? k_geo_bwd<LJ, NH, true, PR, true> : k_geo_bwd<LJ, NH, false, PR, true>;
        }
        AM_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
        {
            KernelTimer kt_("geo_bwd", s);
            hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), lds, s, a, pts, randn, n, table,
                               params, fdv, store, g_sdf, g_grad, g_normal, g_feature, g_laplace,
                               w.genc, w.partial);
        }
        AM_LAUNCH_CHECK();
        return AM_OK;
    };
    if (flag_value("table_atomic", 0) != 0) {
        // atomic form: the pairs are added into the zeroed table gradient
        if (int rc = fill_f32(dtable, (int64_t)g->n_entries * 2, 0.0f, s)) return rc;
        if (int rc = launch_bwd()) return rc;
        if (int rc = pairs_atomic(a, LJ, pts, randn, n, fdv, w.genc, dtable, s)) return rc;
        return colsum_f32(w.partial, waves, a.n_params, dparams, w.ctmp, s);
    }
    // 1. the pairs each part of the emission makes, 2. their prefix sums
    if (int rc = pairs_count(a, LJ, pts, randn, n, fdv, w.pairs, s)) return rc;
    // 3. the pair arrays.  Sync-free form (flag "sdf_bwd_sync_free"): arrays
    // of the worst-case pair bound, no host read (the reduction reads the
    // streams' bounds on the device).  Otherwise one host read of the pair
    // count carves the arrays for exactly that many pairs.  A workspace too
    // small is rejected here, before any output is written, with
    // am_last_workspace_need() = what this call needs.
    const bool bounded = flag_value("sdf_bwd_sync_free", 0) != 0;
    int64_t st[3] = {pairs_bound(a, w.pairs, LJ, n), 0, 0};
    if (!bounded) {
        AM_HIP(hipMemcpyAsync(st, w.pairs.status, sizeof(st), hipMemcpyDeviceToHost, s));
        AM_HIP(hipStreamSynchronize(s));
        timer_units("host_syncs", 1);
    }
    if (int rc = collect_flags(false)) return rc;
    TablePages tp;
    TableReduceWs tw;
    if (int rc = carve_pairs(c, a, g, w.pairs, st[0], &tp, &tw)) return rc;
    if (!c.ok()) return workspace_short(c.used, ws_bytes);
    if (int rc = launch_bwd()) return rc;
    if (int rc = colsum_f32(w.partial, waves, a.n_params, dparams, w.ctmp, s)) return rc;
    if (!bounded) timer_units("table_pairs", st[2]);
    if (int rc = pairs_reduce(a, LJ, g, pts, randn, n, fdv, w.genc, w.pairs, tp, tw, bounded, dtable,
                              s))
        return rc;
    return arm_flag(w.pairs.status + 1, s);
}

template <int LJ, int NH>
static int geo_bwd_launch(const GeoArgs& a, const am_grid_desc* g, const am_mlp_desc* m,
                          const am_sdf_desc* sd, const float* pts, const float* randn, int64_t n,
                          const void* table, const float* params, const float* fdv_in,
                          const float* store, const float* g_sdf, const float* g_grad,
                          const float* g_normal, const float* g_feature, const float* g_laplace,
                          float* dtable, float* dparams, void* ws, size_t ws_bytes, hipStream_t s) {
    if (a.prec == AM_PREC_MIXED)
        return geo_bwd_launch_t<LJ, NH, mlp::kBF16>(a, g, pts, randn, n, table, params, fdv_in,
                                                    store, g_sdf, g_grad, g_normal, g_feature,
                                                    g_laplace, dtable, dparams, ws, ws_bytes, s);
    return geo_bwd_launch_t<LJ, NH, mlp::kF32>(a, g, pts, randn, n, table, params, fdv_in, store,
                                               g_sdf, g_grad, g_normal, g_feature, g_laplace,
                                               dtable, dparams, ws, ws_bytes, s);
}

#define AM_GEO_DISPATCH(FN, ...)                                                   \
    do {                                                                           \
        const bool two = m->n_hidden_layers == 2;                                  \
        switch (LJ) {                                                              \
            case 2: return two ? FN<2, 2>(__VA_ARGS__) : FN<2, 1>(__VA_ARGS__);    \
            default: return two ? FN<4, 2>(__VA_ARGS__) : FN<4, 1>(__VA_ARGS__);   \
        }                                                                          \
    } while (0)

}  // namespace am

using namespace am;

extern "C" int64_t am_sdf_store_floats(const am_grid_desc* g, const am_mlp_desc* m,
                                       const am_sdf_desc* sd, int64_t n) {
    GeoArgs a;
    int LJ;
    if (make_geo_args(g, m, sd, &a, &LJ) || n < 0) return -1;
    const int64_t tiles = (n + 15) / 16;
    return geo_enc_floats(tiles, a.n_evals, LJ) + geo_dx_floats(tiles, a.n_dx, LJ);
}

static int sdf_fwd(const am_grid_desc* g, const am_mlp_desc* m, const am_sdf_desc* sd,
                   const int32_t* order, const float* pts, const float* randn, int64_t n,
                   const void* table, const float* params, float* sdf, float* grad,
                   float* normal, float* feature, float* laplace, float* fd_values,
                   float* enc_store, void* stream) {
    GeoArgs a;
    int LJ;
    if (int rc = make_geo_args(g, m, sd, &a, &LJ)) return rc;
    a.order = order;
    AM_CHECK_ARG(n >= 0, "n < 0");
    if (n == 0) return AM_OK;
    AM_CHECK_ARG(pts && table && params && sdf, "NULL buffer");
    AM_CHECK_ARG(!sd->with_laplace || randn, "laplace needs randn");
    hipStream_t s = to_stream(stream);
    AM_GEO_DISPATCH(geo_fwd_launch, a, pts, randn, n, table, params, sdf, grad, normal, feature,
                    laplace, fd_values, enc_store, s);
}

extern "C" int am_sdf_fwd(const am_grid_desc* g, const am_mlp_desc* m, const am_sdf_desc* sd,
                          const float* pts, const float* randn, int64_t n, const void* table,
                          const float* params, float* sdf, float* grad, float* normal,
                          float* feature, float* laplace, float* fd_values, float* enc_store,
                          void* stream) {
    return sdf_fwd(g, m, sd, nullptr, pts, randn, n, table, params, sdf, grad, normal, feature,
                   laplace, fd_values, enc_store, stream);
}

extern "C" int am_sdf_fwd_ordered(const am_grid_desc* g, const am_mlp_desc* m,
                                  const am_sdf_desc* sd, const int32_t* order, const float* pts,
                                  const float* randn, int64_t n, const void* table,
                                  const float* params, float* sdf, float* grad, float* normal,
                                  float* feature, float* laplace, float* fd_values,
                                  float* enc_store, void* stream) {
    AM_CHECK_ARG(order || n == 0, "NULL order");
    return sdf_fwd(g, m, sd, order, pts, randn, n, table, params, sdf, grad, normal, feature,
                   laplace, fd_values, enc_store, stream);
}

extern "C" size_t am_sdf_bwd_workspace_size(const am_grid_desc* g, const am_mlp_desc* m,
                                            const am_sdf_desc* sd, int64_t n) {
    GeoArgs a;
    int LJ;
    if (make_geo_args(g, m, sd, &a, &LJ) || n < 0) return 0;
    WsCarver c(nullptr, 0);
    GeoBwdWs w;
    carve_geo_bwd_head(c, a, g, LJ, n, true, &w);
    TablePages tp;
    TableReduceWs tw;
    if (carve_pairs(c, a, g, w.pairs, pairs_bound(a, w.pairs, LJ, n), &tp, &tw)) return 0;
    return c.used + 256;
}

extern "C" int am_sdf_bwd_check(void) { return collect_flags(true); }

static int sdf_bwd(const am_grid_desc* g, const am_mlp_desc* m, const am_sdf_desc* sd,
                   const int32_t* order, const float* pts, const float* randn, int64_t n,
                   const void* table, const float* params, const float* fd_values,
                   const float* enc_store, const float* g_sdf, const float* g_grad,
                   const float* g_normal, const float* g_feature, const float* g_laplace,
                   float* dtable, float* dparams, void* workspace, size_t workspace_bytes,
                   void* stream) {
    GeoArgs a;
    int LJ;
    if (int rc = make_geo_args(g, m, sd, &a, &LJ)) return rc;
    a.order = order;
    AM_CHECK_ARG(n >= 0, "n < 0");
    AM_CHECK_ARG(table && params && dtable && dparams && workspace, "NULL buffer");
    hipStream_t s = to_stream(stream);
    if (n == 0) {
        if (int rc = fill_f32(dtable, (int64_t)g->n_entries * 2, 0.0f, s)) return rc;
        return fill_f32(dparams, a.n_params, 0.0f, s);
    }
    AM_CHECK_ARG(pts, "NULL pts");
    AM_CHECK_ARG(!sd->with_laplace || randn, "laplace needs randn");
    AM_GEO_DISPATCH(geo_bwd_launch, a, g, m, sd, pts, randn, n, table, params, fd_values,
                    enc_store, g_sdf, g_grad, g_normal, g_feature, g_laplace, dtable, dparams,
                    workspace, workspace_bytes, s);
}

extern "C" int am_sdf_bwd(const am_grid_desc* g, const am_mlp_desc* m, const am_sdf_desc* sd,
                          const float* pts, const float* randn, int64_t n, const void* table,
                          const float* params, const float* fd_values, const float* enc_store,
                          const float* g_sdf, const float* g_grad, const float* g_normal,
                          const float* g_feature, const float* g_laplace, float* dtable,
                          float* dparams, void* workspace, size_t workspace_bytes, void* stream) {
    return sdf_bwd(g, m, sd, nullptr, pts, randn, n, table, params, fd_values, enc_store, g_sdf,
                   g_grad, g_normal, g_feature, g_laplace, dtable, dparams, workspace,
                   workspace_bytes, stream);
}

extern "C" int am_sdf_bwd_ordered(const am_grid_desc* g, const am_mlp_desc* m,
                                  const am_sdf_desc* sd, const int32_t* order, const float* pts,
                                  const float* randn, int64_t n, const void* table,
                                  const float* params, const float* fd_values,
                                  const float* enc_store, const float* g_sdf, const float* g_grad,
                                  const float* g_normal, const float* g_feature,
                                  const float* g_laplace, float* dtable, float* dparams,
                                  void* workspace, size_t workspace_bytes, void* stream) {
    AM_CHECK_ARG(order || n == 0, "NULL order");
    return sdf_bwd(g, m, sd, order, pts, randn, n, table, params, fd_values, enc_store, g_sdf,
                   g_grad, g_normal, g_feature, g_laplace, dtable, dparams, workspace,
                   workspace_bytes, stream);
}
