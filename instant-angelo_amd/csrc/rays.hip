// Training-ray sampling on the device (systems/neus.py:35-118, train stage):
// per ray k a view v = index[k] and a pixel (y[k], x[k]) drawn by the caller;
// the camera-space direction of that pixel rotated by the view's c2w
// (models/ray_utils.py:23-31: rays_d_i = sum_j d_j c2w[i][j]), normalized as
// F.normalize does (x / max(|x|, 1e-12)); the origin is the c2w translation;
// the pixel's colour and foreground mask gathered, and, when the dataset
// applies masks, blended with the background colour.  Replaces the host-side
// index / gather / get_rays round trip of the reference's preprocess_data.
//
// One lane per ray: the work is a handful of dependent gathers (c2w row
// triplet, a direction, a pixel) and 40 B written per ray.
#include <cmath>
#include "am_common.h"

namespace am {

struct RaySampleArgs {
    const float* images;      // [n_views, H, W, C], C >= 3 (channels 0..2 used)
    const float* fg_masks;    // [n_views, H, W] or nullptr (all foreground)
    const float* c2w;         // [n_views, 3, 4]
    const float* directions;  // [H, W, 3] or [n_views, H, W, 3]
    const float* bg_color;    // [3] device, or nullptr when apply_mask == 0
    int32_t n_views, H, W, C, dirs_per_view, apply_mask;
};

__global__ void k_sample_rays(RaySampleArgs a, const int32_t* __restrict__ index,
                              const int32_t* __restrict__ ys, const int32_t* __restrict__ xs,
                              int64_t n, float* __restrict__ rays, float* __restrict__ rgb,
                              float* __restrict__ fg, int32_t* __restrict__ bad) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int v = index[k], y = ys[k], x = xs[k];
    // out-of-range draws are clamped (no out-of-bounds read) and counted
    if (v < 0 || v >= a.n_views || y < 0 || y >= a.H || x < 0 || x >= a.W) {
        atomicAdd(bad, 1);
        v = min(max(v, 0), a.n_views - 1);
        y = min(max(y, 0), a.H - 1);
        x = min(max(x, 0), a.W - 1);
    }
    const int64_t pix = ((int64_t)v * a.H + y) * a.W + x;
    const int64_t dpix = a.dirs_per_view ? pix : (int64_t)y * a.W + x;
    const float d0 = a.directions[3 * dpix], d1 = a.directions[3 * dpix + 1],
                d2 = a.directions[3 * dpix + 2];
    const float* m = a.c2w + 12 * (int64_t)v;
    float r[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] = (d0 * m[4 * i] + d1 * m[4 * i + 1]) + d2 * m[4 * i + 2];
    const float nrm = sqrtf((r[0] * r[0] + r[1] * r[1]) + r[2] * r[2]);
    const float den = fmaxf(nrm, 1e-12f);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        rays[6 * k + i] = m[4 * i + 3];
        rays[6 * k + 3 + i] = r[i] / den;
    }
    const float f = a.fg_masks ? a.fg_masks[pix] : 1.0f;
    const float* px = a.images + pix * a.C;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        float c = px[i];
        if (a.apply_mask) c = c * f + a.bg_color[i] * (1.0f - f);
        rgb[3 * k + i] = c;
    }
    fg[k] = f;
}

// Morton (Z-order) key of a sample: its position in [-r, r]^3 quantised to
// `bits` (<= 10) bits per axis and the bits interleaved (x highest).  Sorting samples by
// it makes the waves that run together gather nearby table rows.
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t morton_key(const float* __restrict__ pts, int64_t i, float r,
                                               float inv2r, int bits) {
    const uint32_t cells = 1u << bits;
    uint32_t q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        float u = (pts[3 * i + d] + r) * inv2r;
        u = fminf(fmaxf(u, 0.0f), 1.0f);   // NaN -> 0
        const uint32_t v = (uint32_t)(u * (float)cells);
        q[d] = v > cells - 1 ? cells - 1 : v;
    }
    return (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
}

__global__ void k_morton_keys(const float* __restrict__ pts, int64_t n, float r, float inv2r,
                              int bits, int32_t* __restrict__ keys) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = (int32_t)morton_key(pts, i, r, inv2r, bits);
}

// Stable order by key: least-significant-digit counting passes of up to 8 bits
// (15-bit keys: two), each a digit histogram per block and a scatter.  At most
// kOrderBlocks blocks of whole 1024-sample tiles, so that every scatter block
// sums the histograms before its own by itself: no scan between the two, and
// four launches in all for 15-bit keys.  Bound by launches and by the chain of
// passes at 65 k samples, by the scattered writes at 1 M.  A merge sort of the
// same keys (one launch a doubling), with its key, index and inverse kernels:
// 65 k samples 43 -> 22 us, 262 k 99 -> 25, 940 k 169 -> 45, 4.8 M 230 -> 150.
// Twice the blocks above kOrderWide samples, where a block a CU no longer
// covers its loads' latency (60 M samples, 30-bit keys 3298 -> 2979 us, the sort
// 2947; 20 M 1049 -> 968).
constexpr int kOrderTile = 1024;     // samples a tile: one a thread
constexpr int kOrderBlocks = 256;
constexpr int64_t kOrderWide = 1 << 24;
constexpr int kDigits = 256;
static inline int64_t order_blocks(int64_t n) {
    return n > kOrderWide ? 2 * kOrderBlocks : kOrderBlocks;
}

struct OrderPass {
    const float* pts;      // first pass: keys from the positions
    float r, inv2r;
    int bits;
    const uint2* in;       // later passes: (key, sample)
    uint2* out;            // all but the last
    int32_t* perm;         // the last
    int32_t* inv;
    int shift, width;
    int64_t n;
    int tiles;             // tiles a block
};

template <bool FIRST>
__device__ __forceinline__ uint2 order_item(const OrderPass& a, int64_t i) {
    if constexpr (FIRST) return make_uint2(morton_key(a.pts, i, a.r, a.inv2r, a.bits), (uint32_t)i);
    else return a.in[i];
}

template <bool FIRST>
__global__ void __launch_bounds__(kOrderTile) k_order_hist(OrderPass a,
                                                           uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[kDigits];
    const int tid = (int)threadIdx.x;
    if (tid < kDigits) h[tid] = 0u;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * a.tiles * kOrderTile;
    for (int t = 0; t < a.tiles; ++t) {
        const int64_t i = first + (int64_t)t * kOrderTile + tid;
        if (i < a.n)
            atomicAdd(&h[order_item<FIRST>(a, i).x >> a.shift & ((1u << a.width) - 1u)], 1u);
    }
    __syncthreads();
    if (tid < kDigits) hist[(int64_t)blockIdx.x * kDigits + tid] = h[tid];
}

// The wave's lanes with this lane's digit, and how many of them lie before it.
__device__ __forceinline__ int digit_rank(bool on, uint32_t digit, uint64_t* lanes) {
    uint64_t same = __ballot(on);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = digit >> b & 1u;
        const uint64_t set = __ballot(bit);
        same &= bit ? set : ~set;
    }
    *lanes = same;
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
}

template <bool FIRST, bool LAST>
__global__ void __launch_bounds__(kOrderTile) k_order_scatter(OrderPass a,
                                                              const uint32_t* __restrict__ hist) {
    __shared__ uint32_t count[kOrderTile / 64][kDigits];   // a tile's, per wave; its places
    __shared__ uint32_t before[4][kDigits], total[4][kDigits];
    __shared__ uint32_t place[kDigits];                    // next position of each digit
    __shared__ uint32_t wave_sum[4];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the digits' totals, and what earlier blocks put before this one's
    {
        const int d = tid & (kDigits - 1), q = tid >> 8;
        uint32_t sum = 0, mine = 0;
#pragma unroll 8
        for (int b = q; b < (int)gridDim.x; b += 4) {
            const uint32_t v = hist[(int64_t)b * kDigits + d];
            sum += v;
            mine += b < (int)blockIdx.x ? v : 0u;
        }
        total[q][d] = sum;
        before[q][d] = mine;
    }
    for (int q = tid; q < (kOrderTile / 64) * kDigits; q += kOrderTile) (&count[0][0])[q] = 0u;
    __syncthreads();
    uint32_t all = 0, incl = 0;
    if (tid < kDigits) {
        all = (total[0][tid] + total[1][tid]) + (total[2][tid] + total[3][tid]);
        incl = all;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            const uint32_t o = __shfl_up(incl, s, 64);
            if (lane >= s) incl += o;
        }
        if (lane == 63) wave_sum[wave] = incl;
    }
    __syncthreads();
    if (tid < kDigits) {
        uint32_t at = incl - all;
#pragma unroll
        for (int w = 0; w < 4; ++w) at += w < wave ? wave_sum[w] : 0u;
        place[tid] = at + (before[0][tid] + before[1][tid]) + (before[2][tid] + before[3][tid]);
    }
    const int64_t first = (int64_t)blockIdx.x * a.tiles * kOrderTile;
    for (int t = 0; t < a.tiles; ++t) {
        const int64_t i = first + (int64_t)t * kOrderTile + tid;
        const bool on = i < a.n;
        const uint2 it = on ? order_item<FIRST>(a, i) : make_uint2(0u, 0u);
        const uint32_t digit = it.x >> a.shift & ((1u << a.width) - 1u);
        uint64_t same;
        const int rank = digit_rank(on, digit, &same);
        if (on && rank == 0) count[wave][digit] = (uint32_t)__popcll(same);
        __syncthreads();
        if (tid < kDigits) {   // counts to places, waves in order
            uint32_t at = place[tid];
#pragma unroll
            for (int w = 0; w < kOrderTile / 64; ++w) {
                const uint32_t c = count[w][tid];
                count[w][tid] = at;
                at += c;
            }
            place[tid] = at;
        }
        __syncthreads();
        if (on) {
            const uint32_t to = count[wave][digit] + (uint32_t)rank;
            if constexpr (LAST) {
                a.perm[to] = (int32_t)it.y;
                a.inv[it.y] = (int32_t)to;
            } else {
                a.out[to] = it;
            }
        }
        if (t + 1 < a.tiles) {
            __syncthreads();
            for (int q = tid; q < (kOrderTile / 64) * kDigits; q += kOrderTile)
                (&count[0][0])[q] = 0u;
            __syncthreads();
        }
    }
}

// All passes of up to kOrderOne samples in one block and one launch, the samples
// in LDS between passes: bound by that launch (1000 samples, 15- and 30-bit keys
// 16 us, two launches a pass 24 and 36, the sort 27; 4096 samples 16 and 26
// against 25 and 36, the sort 32).
constexpr int kOneTiles = 4;
constexpr int kOrderOne = kOneTiles * kOrderTile;

__global__ void __launch_bounds__(kOrderTile) k_order_one(OrderPass a, int passes) {
    __shared__ uint2 items[kOrderOne];
    __shared__ uint32_t count[kOrderTile / 64][kDigits];   // a tile's, per wave; its places
    __shared__ uint32_t place[kDigits];
    __shared__ uint32_t wave_sum[4];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = (int)a.n, tiles = (n + kOrderTile - 1) / kOrderTile;
    uint2 it[kOneTiles];
#pragma unroll
    for (int t = 0; t < kOneTiles; ++t) {
        const int i = t * kOrderTile + tid;
        it[t] = i < n ? order_item<true>(a, i) : make_uint2(0u, 0u);
    }
    for (int p = 0; p < passes; ++p) {
        const int shift = p * a.width;
        const uint32_t mask = (1u << a.width) - 1u;
        if (tid < kDigits) place[tid] = 0u;
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kOneTiles; ++t)
            if (t * kOrderTile + tid < n) atomicAdd(&place[it[t].x >> shift & mask], 1u);
        __syncthreads();
        uint32_t all = 0, incl = 0;
        if (tid < kDigits) {
            incl = all = place[tid];
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) {
                const uint32_t o = __shfl_up(incl, s, 64);
                if (lane >= s) incl += o;
            }
            if (lane == 63) wave_sum[wave] = incl;
        }
        __syncthreads();
        if (tid < kDigits) {
            uint32_t at = incl - all;
#pragma unroll
            for (int w = 0; w < 4; ++w) at += w < wave ? wave_sum[w] : 0u;
            place[tid] = at;
        }
#pragma unroll
        for (int t = 0; t < kOneTiles; ++t) {
            if (t >= tiles) break;
            for (int q = tid; q < (kOrderTile / 64) * kDigits; q += kOrderTile) (&count[0][0])[q] = 0u;
            __syncthreads();
            const bool on = t * kOrderTile + tid < n;
            const uint32_t digit = it[t].x >> shift & mask;
            uint64_t same;
            const int rank = digit_rank(on, digit, &same);
            if (on && rank == 0) count[wave][digit] = (uint32_t)__popcll(same);
            __syncthreads();
            if (tid < kDigits) {   // counts to places, waves in order
                uint32_t at = place[tid];
#pragma unroll
                for (int w = 0; w < kOrderTile / 64; ++w) {
                    const uint32_t c = count[w][tid];
                    count[w][tid] = at;
                    at += c;
                }
                place[tid] = at;
            }
            __syncthreads();
            if (on) {
                const uint32_t to = count[wave][digit] + (uint32_t)rank;
                if (p + 1 < passes) items[to] = it[t];
                else {
                    a.perm[to] = (int32_t)it[t].y;
                    a.inv[it[t].y] = (int32_t)to;
                }
            }
            __syncthreads();
        }
        if (p + 1 < passes) {
#pragma unroll
            for (int t = 0; t < kOneTiles; ++t)
                if (t * kOrderTile + tid < n) it[t] = items[t * kOrderTile + tid];
            __syncthreads();
        }
    }
}

}  // namespace am

using namespace am;

extern "C" size_t am_morton_order_workspace_size(int64_t n, int32_t bits) {
    if (n < 0 || bits < 1 || bits > 10) return 0;
    WsCarver c(nullptr, 0);
    c.take<uint32_t>((size_t)order_blocks(n) * kDigits);
    for (int b = 0; b < 2; ++b) c.take<uint2>((size_t)n + 1);
    return c.used + 256;
}

extern "C" int am_morton_order(const float* pts, int64_t n, float radius, int32_t bits,
                               int32_t* perm, int32_t* inv, void* workspace,
                               size_t workspace_bytes, void* stream) {
    AM_CHECK_ARG(n >= 0 && n < (1ll << 31), "n %lld", (long long)n);
    AM_CHECK_ARG(radius > 0.0f, "radius %g <= 0", (double)radius);
    AM_CHECK_ARG(bits >= 1 && bits <= 10, "bits %d out of [1, 10]", bits);
    if (n == 0) return AM_OK;
    AM_CHECK_ARG(pts && perm && inv && workspace, "NULL buffer");
    hipStream_t s = to_stream(stream);
    WsCarver c(workspace, workspace_bytes);
    uint32_t* hist = c.take<uint32_t>((size_t)order_blocks(n) * kDigits);
    uint2* items[2];
    for (int b = 0; b < 2; ++b) items[b] = c.take<uint2>((size_t)n + 1);
    if (!c.ok()) return workspace_short(c.used, workspace_bytes);
    const int64_t all_tiles = ceil_div(n, kOrderTile);
    const int passes = (3 * bits + 7) / 8, width = (3 * bits + passes - 1) / passes;
    OrderPass a{};
    a.pts = pts;
    a.r = radius;
    a.inv2r = 0.5f / radius;
    a.bits = bits;
    a.perm = perm;
    a.inv = inv;
    a.width = width;
    a.n = n;
    a.tiles = (int)ceil_div(all_tiles, order_blocks(n));
    const unsigned nb = (unsigned)ceil_div(all_tiles, a.tiles);
    if (n <= kOrderOne) {
        hipLaunchKernelGGL(k_order_one, dim3(1), dim3(kOrderTile), 0, s, a, passes);
        AM_LAUNCH_CHECK();
        return AM_OK;
    }
    for (int p = 0; p < passes; ++p) {
        const bool last = p == passes - 1;
        a.shift = p * width;
        a.in = items[(p + 1) & 1];
        a.out = items[p & 1];
        auto hist_kern = p == 0 ? k_order_hist<true> : k_order_hist<false>;
        auto kern = p == 0 ? (last ? k_order_scatter<true, true> : k_order_scatter<true, false>)
                           : (last ? k_order_scatter<false, true> : k_order_scatter<false, false>);
        hipLaunchKernelGGL(hist_kern, dim3(nb), dim3(kOrderTile), 0, s, a, hist);
        AM_LAUNCH_CHECK();
        hipLaunchKernelGGL(kern, dim3(nb), dim3(kOrderTile), 0, s, a, hist);
        AM_LAUNCH_CHECK();
    }
    return AM_OK;
}

extern "C" int am_morton_keys(const float* pts, int64_t n, float radius, int32_t* keys,
                              void* stream) {
    AM_CHECK_ARG(n >= 0, "n < 0");
    AM_CHECK_ARG(radius > 0.0f, "radius %g <= 0", (double)radius);
    if (n == 0) return AM_OK;
    AM_CHECK_ARG(pts && keys, "NULL buffer");
    hipLaunchKernelGGL(k_morton_keys, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0,
                       to_stream(stream), pts, n, radius, 0.5f / radius, 10, keys);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

extern "C" int am_sample_rays(const float* images, const float* fg_masks, const float* c2w,
                              const float* directions, int32_t n_views, int32_t H, int32_t W,
                              int32_t C, int32_t dirs_per_view, const float* bg_color,
                              int32_t apply_mask, const int32_t* index, const int32_t* ys,
                              const int32_t* xs, int64_t n, float* rays, float* rgb,
                              float* fg_mask, int32_t* n_out_of_range, void* stream) {
    AM_CHECK_ARG(n >= 0, "n < 0");
    AM_CHECK_ARG(n_views >= 1 && H >= 1 && W >= 1, "empty image set (%d views, %dx%d)", n_views,
                 W, H);
    AM_CHECK_ARG(C >= 3, "images need at least 3 channels (got %d)", C);
    AM_CHECK_ARG(!apply_mask || bg_color, "apply_mask needs bg_color");
    AM_CHECK_ARG((int64_t)n_views * H * W < (1ll << 40), "image set too large");
    if (n == 0) return AM_OK;
    AM_CHECK_ARG(images && c2w && directions && index && ys && xs && rays && rgb && fg_mask &&
                     n_out_of_range, "NULL buffer");
    RaySampleArgs a;
    a.images = images;
    a.fg_masks = fg_masks;
    a.c2w = c2w;
    a.directions = directions;
    a.bg_color = bg_color;
    a.n_views = n_views;
    a.H = H;
    a.W = W;
    a.C = C;
    a.dirs_per_view = dirs_per_view ? 1 : 0;
    a.apply_mask = apply_mask ? 1 : 0;
    {
        KernelTimer kt_("sample_rays", to_stream(stream));
        hipLaunchKernelGGL(k_sample_rays, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0,
                           to_stream(stream), a, index, ys, xs, n, rays, rgb, fg_mask,
                           n_out_of_range);
    }
    AM_LAUNCH_CHECK();
    return AM_OK;
}
