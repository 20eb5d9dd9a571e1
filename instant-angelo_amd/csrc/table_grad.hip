// Deterministic table-gradient reduction: the paged form, and the stable
// radix sort with a fixed-order segmented reduce (see table_grad.h).
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include "page_dev.h"

namespace am {

constexpr int64_t kUnitItems = 16384;   // sorted items per work unit (256 chunks)

// Partial-sum slots the units of multi-unit buckets can need: each such
// bucket holds more than kUnitItems items and fewer than 2n / kUnitItems units.
static int64_t bucket_slots(int64_t m) { return 2 * (m / kUnitItems) + 1; }

// ---- paged form ----
// Pairs of a work unit: a level's buckets are cut into slices of about this
// many pairs where they hold more (coarse levels), fewer when the whole
// gradient makes less than about 1024 units of the most.
constexpr int64_t kUnitMost = 1 << 19;
constexpr int64_t kUnitLeast = 16384;

// The buckets of a level are written whole and row 0 on to n_entries by the
// levels together, so the levels must follow one another as am_grid_init lays
// them; descriptors with gaps, shared rows or another order take the sorted
// form, which knows rows alone.
bool table_paged(const am_grid_desc* g) {
    if (g->n_features != 2) return false;
    uint64_t next = 0;
    for (int l = 0; l < g->n_levels; ++l) {
        if (g->offset[l] != next || g->size[l] == 0u ||
            g->size[l] > (uint32_t)kMaxDigits * kRows)
            return false;
        next += g->size[l];
    }
    return next == g->n_entries;
}

TableLevels table_levels(const am_grid_desc* g) {
    TableLevels t{};
    t.L = g->n_levels;
    for (int l = 0; l < g->n_levels; ++l) {
        t.offset[l] = g->offset[l];
        t.offset[l + 1] = g->offset[l] + g->size[l];
    }
    return t;
}

// Units of sliced levels: a level of n pairs and D buckets has
// S = ceil(n / (D U)) slices, D S <= 2 n / U where S > 1.
static int64_t slot_bound(int64_t m) {
    const int64_t a = 2 * (m / kUnitLeast), b = 2 * (m / kUnitMost);
    return (a < 2048 ? a : (b > 2048 ? b : 2048)) + 2;
}

static int64_t table_digits(const am_grid_desc* g) {
    int64_t d = 0;
    for (int l = 0; l < g->n_levels; ++l) d += ceil_div(g->size[l], kRows);
    return d;
}

int table_key_bits(uint32_t n_entries) {
    int b = 1;
    while (b < 32 && (1ull << b) <= (uint64_t)n_entries) ++b;
    return b;
}

// Bucketed form: up to 9 low key bits stay unsorted.  Keys of up to 25 bits
// sort their high bits [9, end) in one or two 8-bit onesweep passes (the
// fastest form measured for 16 bits: 8-bit digits rank with less LDS than
// 9-bit ones); 26-27-bit keys in two 9-bit passes, longer ones in three.
int table_bucket_bits(int end_bit) {
    if (end_bit <= 9) return 0;
    if (end_bit <= 25) return 9;
    const int passes = (end_bit - 9 + 8) / 9;
    return end_bit - 9 * passes;
}

static int digit_bits(const TableReduceWs& w) {
    return (w.n_buckets > 0 && w.begin_bit == 9) ? 8 : 9;
}

// Onesweep configurations: 1024-thread blocks of 8 items per thread for the
// sort passes, 32 items per thread for the histogram pass.
using Sort9Config = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<1024, 32>,
                                        rocprim::kernel_config<1024, 8>, 9,
                                        rocprim::block_radix_rank_algorithm::match>>;
using Sort8Config = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<1024, 32>,
                                        rocprim::kernel_config<1024, 8>, 8,
                                        rocprim::block_radix_rank_algorithm::match>>;

template <class VT>
static hipError_t sort_pairs(void* tmp, size_t& bytes, TableReduceWs& w, uint32_t** kout,
                             VT** vout, hipStream_t s) {
    rocprim::double_buffer<uint32_t> kb(w.keys[0], w.keys[1]);
    rocprim::double_buffer<VT> vb(reinterpret_cast<VT*>(w.vals[0]), reinterpret_cast<VT*>(w.vals[1]));
    hipError_t e;
    if (w.n_buckets > 0 && digit_bits(w) == 8)
        e = rocprim::radix_sort_pairs<Sort8Config>(tmp, bytes, kb, vb, (size_t)w.m,
                                                   (unsigned)w.begin_bit, (unsigned)w.end_bit, s,
                                                   false);
    else if (w.n_buckets > 0 || (w.end_bit > 24 && w.end_bit <= 27))
        e = rocprim::radix_sort_pairs<Sort9Config>(tmp, bytes, kb, vb, (size_t)w.m,
                                                   (unsigned)w.begin_bit, (unsigned)w.end_bit, s,
                                                   false);
    else
        e = rocprim::radix_sort_pairs(tmp, bytes, kb, vb, (size_t)w.m, 0u, (unsigned)w.end_bit, s,
                                      false);
    if (kout) *kout = kb.current();
    if (vout) *vout = vb.current();
    return e;
}

int table_reduce_carve(WsCarver& c, const am_grid_desc* g, int64_t m, TableReduceWs* out,
                       bool half_vals) {
    const int F = g->n_features;
    const uint32_t n_entries = g->n_entries;
    TableReduceWs w{};
    w.m = m;
    w.end_bit = table_key_bits(n_entries);
    w.half_vals = half_vals;
    const size_t vbytes = (size_t)F * (half_vals ? sizeof(__half) : sizeof(float));
    w.keys[0] = c.take<uint32_t>((size_t)m);
    w.keys[1] = c.take<uint32_t>((size_t)m);
    w.vals[0] = c.take<char>((size_t)m * vbytes);
    w.vals[1] = c.take<char>((size_t)m * vbytes);
    if (F == 2) {   // bucketed form
        w.begin_bit = table_bucket_bits(w.end_bit);
        w.n_buckets = ceil_div((int64_t)n_entries, (int64_t)1 << w.begin_bit);
        w.bucket_start = c.take<int64_t>((size_t)w.n_buckets + 1);
        w.units = c.take<uint64_t>((size_t)w.n_buckets + 1);
        w.unit_off = c.take<uint64_t>((size_t)w.n_buckets + 1);
        w.partial = c.take<float>((size_t)bucket_slots(m) * (2u << w.begin_bit));
        size_t scb = 0;
        if (rocprim::exclusive_scan(nullptr, scb, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                    (uint64_t)0, (size_t)w.n_buckets + 1,
                                    rocprim::plus<uint64_t>(), 0, false) != hipSuccess) {
            set_error("bucket unit scan size query failed");
            return AM_ERR_HIP;
        }
        w.scan_bytes = scb;
        w.scan_tmp = c.take<char>(scb + 256);
    } else {        // chunked segmented reduce
        const int64_t nc = ceil_div(m, kSegChunk);
        w.lead = c.take<float>((size_t)nc * F);
        w.tail = c.take<float>((size_t)nc * F);
        w.lead_full = c.take<uint8_t>((size_t)nc);
        w.tail_open = c.take<uint8_t>((size_t)nc);
    }
    size_t sb = 0;
    hipError_t e = hipSuccess;
    if (half_vals && F != 2) {
        set_error("fp16 gradient pairs need n_features = 2 (got %d)", F);
        return AM_ERR_UNSUPPORTED;
    }
    switch (half_vals ? -F : F) {
        case 1: e = sort_pairs<Vals<1>>(nullptr, sb, w, nullptr, nullptr, 0); break;
        case 2: e = sort_pairs<Vals<2>>(nullptr, sb, w, nullptr, nullptr, 0); break;
        case 4: e = sort_pairs<Vals<4>>(nullptr, sb, w, nullptr, nullptr, 0); break;
        case 8: e = sort_pairs<Vals<8>>(nullptr, sb, w, nullptr, nullptr, 0); break;
        case -2: e = sort_pairs<ValsH<2>>(nullptr, sb, w, nullptr, nullptr, 0); break;
        default: set_error("unsupported n_features %d", F); return AM_ERR_UNSUPPORTED;
    }
    if (e != hipSuccess) {
        set_error("radix sort size query failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    w.sort_bytes = sb;
    w.sort_tmp = c.take<char>(sb + 256);
    *out = w;
    return AM_OK;
}

__global__ void k_fill_f32(float* __restrict__ p, int64_t n, float v) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Pass A: each thread reduces kSegChunk consecutive sorted items.  Segments
// wholly inside the chunk are written; the piece continuing a segment from the
// previous chunk goes to lead[t] (lead_full: the chunk is entirely that piece
// and the segment goes on); a segment starting here and continuing goes to
// tail[t] (tail_open).  The block first stages its 256 chunks through LDS
// with coalesced loads (kSegChunk is odd, so per-thread LDS strides spread
// over the banks).
template <int F>
struct SegCfg {
    static constexpr int threads = F <= 2 ? 256 : 64;
};

template <int F, class VT>
__global__ void __launch_bounds__(SegCfg<F>::threads) k_seg_a(
    const uint32_t* __restrict__ keys, const VT* __restrict__ vals, int64_t m,
    uint32_t n_entries, float* __restrict__ out, float* __restrict__ lead,
    float* __restrict__ tail, uint8_t* __restrict__ lead_full, uint8_t* __restrict__ tail_open) {
    constexpr int kSegThreads = SegCfg<F>::threads;
    __shared__ uint32_t sk[kSegThreads * kSegChunk + 1];
    __shared__ float sv[kSegThreads * kSegChunk * F];
    const int64_t blk0 = (int64_t)blockIdx.x * kSegThreads * kSegChunk;
    const int64_t blk_n = m - blk0 < (int64_t)kSegThreads * kSegChunk ? m - blk0
                                                                     : (int64_t)kSegThreads * kSegChunk;
    for (int q = threadIdx.x; q < blk_n; q += kSegThreads) sk[q] = keys[blk0 + q];
    if constexpr (sizeof(VT) == F * sizeof(float)) {
        const float* vf = reinterpret_cast<const float*>(vals) + blk0 * F;
        for (int q = threadIdx.x; q < blk_n * F; q += kSegThreads) sv[q] = vf[q];
    } else {
        const __half* vh = reinterpret_cast<const __half*>(vals) + blk0 * F;
        for (int q = threadIdx.x; q < blk_n * F; q += kSegThreads) sv[q] = __half2float(vh[q]);
    }
    __syncthreads();
    const int64_t t = (int64_t)blockIdx.x * kSegThreads + threadIdx.x;
    const int64_t nc = (m + kSegChunk - 1) / kSegChunk;
    if (t >= nc) return;
    const int lb = threadIdx.x * kSegChunk;                 // local begin
    const int64_t b = t * kSegChunk;
    const int64_t e = b + kSegChunk < m ? b + kSegChunk : m;
    const int le = lb + (int)(e - b);
    bool is_lead = b > 0 && sk[lb] == (lb > 0 ? sk[lb - 1] : keys[b - 1]);
    uint32_t cur = sk[lb];
    float acc[F];
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = 0.0f;
    for (int j = lb; j < le; ++j) {
        const uint32_t k = sk[j];
        if (k != cur) {
            if (is_lead) {
#pragma unroll
                for (int f = 0; f < F; ++f) lead[t * F + f] = acc[f];
                is_lead = false;
            } else if (cur < n_entries) {
#pragma unroll
                for (int f = 0; f < F; ++f) out[(int64_t)cur * F + f] = acc[f];
            }
            cur = k;
#pragma unroll
            for (int f = 0; f < F; ++f) acc[f] = 0.0f;
        }
#pragma unroll
        for (int f = 0; f < F; ++f) acc[f] += sv[j * F + f];
    }
    const bool cont_out = e < m && keys[e] == cur;
    uint8_t lf = 0, to = 0;
    if (is_lead) {
#pragma unroll
        for (int f = 0; f < F; ++f) lead[t * F + f] = acc[f];
        lf = cont_out ? 1 : 0;
    } else if (cont_out) {
#pragma unroll
        for (int f = 0; f < F; ++f) tail[t * F + f] = acc[f];
        to = 1;
    } else if (cur < n_entries) {
#pragma unroll
        for (int f = 0; f < F; ++f) out[(int64_t)cur * F + f] = acc[f];
    }
    lead_full[t] = lf;
    tail_open[t] = to;
}

// Pass B: a segment spanning chunks is summed by the chunk it starts in:
// its tail piece, then each following chunk's lead piece, in chunk order.
template <int F>
__global__ void k_seg_b(const uint32_t* __restrict__ keys, int64_t m, uint32_t n_entries,
                        float* __restrict__ out, const float* __restrict__ lead,
                        const float* __restrict__ tail, const uint8_t* __restrict__ lead_full,
                        const uint8_t* __restrict__ tail_open) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nc = (m + kSegChunk - 1) / kSegChunk;
    if (t >= nc || !tail_open[t]) return;
    const int64_t last = (t + 1) * kSegChunk - 1;
    const uint32_t key = keys[last];
    if (key >= n_entries) return;
    float acc[F];
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = tail[t * F + f];
    for (int64_t u = t + 1; u < nc; ++u) {
#pragma unroll
        for (int f = 0; f < F; ++f) acc[f] += lead[u * F + f];
        if (!lead_full[u]) break;
    }
#pragma unroll
    for (int f = 0; f < F; ++f) out[(int64_t)key * F + f] = acc[f];
}

// Bucketed form.  start[k] = first sorted item of bucket k (keys sorted on
// bits >= B, so key >> B is non-decreasing), k in [0, n_buckets].
__global__ void k_bucket_bounds(const uint32_t* __restrict__ keys, int64_t m, int B,
                                int64_t n_buckets, int64_t* __restrict__ start) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t > n_buckets) return;
    // start[n_buckets] is searched too: sentinel keys of empty slots may
    // lie past the last bucket and must stay out of its range
    int64_t lo = 0, hi = m;
    while (lo < hi) {
        const int64_t mid = lo + ((hi - lo) >> 1);
        if ((int64_t)(keys[mid] >> B) < t) lo = mid + 1;
        else hi = mid;
    }
    start[t] = lo;
}

__device__ __forceinline__ int popc_below(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// One round of a stable split of the wave's 64 keys on bit 6 + `bit`: lanes
// with the bit clear keep their order at the front (destination = clear
// lanes below), set ones follow (all clear lanes + set lanes below).
// Branch-free: both destinations come from one count of set lanes below.
__device__ __forceinline__ uint32_t split_round(uint32_t rk, int bit, int lane) {
    const bool one = (rk >> (6 + bit)) & 1u;
    const uint64_t ones = __ballot(one);
    const int below = popc_below(ones);
    const int dst = one ? (64 - (int)__popcll(ones)) + below : lane - below;
    return (uint32_t)__builtin_amdgcn_ds_permute(dst * 4, (int)rk);
}

__device__ __forceinline__ float permute_f(int dst_byte, float v) {
    return __int_as_float(__builtin_amdgcn_ds_permute(dst_byte, __float_as_int(v)));
}

__device__ __forceinline__ float bpermute_f(int src_byte, float v) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src_byte, __float_as_int(v)));
}

__device__ __forceinline__ void load_pair(const Vals<2>* v, int64_t i, float& a, float& b) {
    const float2 x = *reinterpret_cast<const float2*>(v + i);
    a = x.x;
    b = x.y;
}

__device__ __forceinline__ void load_pair(const ValsH<2>* v, int64_t i, float& a, float& b) {
    const __half2 x = *reinterpret_cast<const __half2*>(v + i);
    a = __low2float(x);
    b = __high2float(x);
}

// One step of a segmented inclusive scan over lanes sorted by r: the DPP
// source lane's partial is added when it holds the same row (lanes whose
// source is outside the row, or whose row the mask excludes, read the
// never-matching sentinel).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void seg_step(uint32_t r, float& a, float& b) {
    const uint32_t rs = (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffffu, (int)r, CTRL,
                                                              ROW_MASK, 0xf, false);
    const float as = __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(a), CTRL, ROW_MASK, 0xf, false));
    const float bs = __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(b), CTRL, ROW_MASK, 0xf, false));
    if (rs == r) {
        a += as;
        b += bs;
    }
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kBucketWaves = 4;
constexpr int kMaxBucketBits = 9;

// Work units: a bucket of n items is cut into max(1, ceil(n / kUnitItems))
// consecutive ranges, so a bucket of a coarse (dense, heavily shared) level
// is spread over many waves.  units[b] packs the bucket's unit count (low 32
// bits) and, for a bucket of several units, the same count again (high 32
// bits: its partial-sum slots); an exclusive scan of the packed words gives
// each bucket's first unit and first slot at once.  units[n_buckets] = 0, so
// the scan's last entry holds the totals.
__global__ void k_bucket_units(const int64_t* __restrict__ start, int64_t n_buckets,
                               uint64_t* __restrict__ units) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t > n_buckets) return;
    uint64_t v = 0;
    if (t < n_buckets) {
        const int64_t n = start[t + 1] - start[t];
        const uint64_t ns = n <= kUnitItems ? 1u : (uint64_t)((n + kUnitItems - 1) / kUnitItems);
        v = ns | (ns > 1 ? ns << 32 : 0);
    }
    units[t] = v;
}

// Reduces sorted items [s, e) of one bucket into the wave's LDS accumulators
// acc[2 << B].  Each chunk of 64 items (in emission order) is stable-sorted
// in registers by its row within the bucket (B split rounds of ballot +
// permute; a partial chunk sorts one more bit that moves its empty lanes
// last), reduced by a segmented inclusive scan (DPP row shifts and
// broadcasts: a fixed tree per segment), and each segment's total is added
// to the row's accumulator by the segment's last lane (rows are unique per
// chunk, chunks go in order): the summation order is a fixed function of the
// sorted input.
template <class VT>
__device__ __forceinline__ void reduce_range(const uint32_t* __restrict__ keys,
                                             const VT* __restrict__ vals, int64_t s, int64_t e,
                                             int B, float* acc) {
    const int lane = threadIdx.x & 63;
    const int rows = 1 << B;
    uint32_t nk = 0;
    float na = 0.0f, nb = 0.0f;
    if (s + lane < e) {
        nk = keys[s + lane];
        load_pair(vals, s + lane, na, nb);
    }
    for (int64_t c = s; c < e; c += 64) {
        const bool valid = c + lane < e;
        const uint32_t r0 = valid ? (nk & (uint32_t)(rows - 1)) : (uint32_t)rows;
        const float a0 = valid ? na : 0.0f, b0 = valid ? nb : 0.0f;
        if (c + 64 + lane < e) {   // prefetch the next chunk
            nk = keys[c + 64 + lane];
            load_pair(vals, c + 64 + lane, na, nb);
        }
        // stable split sort of (row << 6 | source lane): one permute per
        // round; the values follow once at the end.  A partial chunk sorts
        // one more bit (its idle lanes carry row `rows`).
        uint32_t rk = (r0 << 6) | (uint32_t)lane;
        if (B == 9) {   // the bucketed sort's digit: unrolled
#pragma unroll
            for (int bit = 0; bit < 9; ++bit) rk = split_round(rk, bit, lane);
            if (e - c < 64) rk = split_round(rk, 9, lane);
        } else {
            const int nbits = (e - c < 64) ? B + 1 : B;
            for (int bit = 0; bit < nbits; ++bit) rk = split_round(rk, bit, lane);
        }
        const uint32_t r = rk >> 6;
        const int from = (int)(rk & 63u) * 4;
        float a = bpermute_f(from, a0);
        float b = bpermute_f(from, b0);
        // segmented inclusive scan over the sorted lanes: row shifts of
        // 1, 2, 4, 8 within 16-lane rows, then the last lane of row 0
        // (row 2) into row 1 (row 3), then lane 31 into rows 2 and 3
        seg_step<0x111, 0xf>(r, a, b);
        seg_step<0x112, 0xf>(r, a, b);
        seg_step<0x114, 0xf>(r, a, b);
        seg_step<0x118, 0xf>(r, a, b);
        seg_step<0x142, 0xa>(r, a, b);
        seg_step<0x143, 0xc>(r, a, b);
        const uint32_t rn = (uint32_t)__builtin_amdgcn_ds_bpermute(((lane + 1) & 63) * 4, (int)r);
        if ((lane == 63 || rn != r) && r < (uint32_t)rows) {
            acc[2 * r] += a;
            acc[2 * r + 1] += b;
        }
        wave_lds_sync();
    }
}

// One wave per work unit (grid-stride).  A single-unit bucket writes its
// rows to dtable, zeros included (dtable needs no fill); a unit of a
// multi-unit bucket writes its accumulators to its partial slot.
template <class VT>
__global__ void __launch_bounds__(64 * kBucketWaves) k_bucket_reduce(
    const uint32_t* __restrict__ keys, const VT* __restrict__ vals,
    const int64_t* __restrict__ start, const uint64_t* __restrict__ uoff, int64_t n_buckets,
    int B, uint32_t n_entries, float* __restrict__ out, float* __restrict__ partial) {
    __shared__ float acc_s[kBucketWaves][2 << kMaxBucketBits];
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    float* acc = acc_s[wave];
    const int rows = 1 << B;
    const int64_t total = (int64_t)(uint32_t)uoff[n_buckets];
    for (int64_t u = (int64_t)blockIdx.x * kBucketWaves + wave; u < total;
         u += (int64_t)gridDim.x * kBucketWaves) {
        // the bucket: the last b with first unit <= u
        int64_t lo = 0, hi = n_buckets - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if ((int64_t)(uint32_t)uoff[mid] <= u) lo = mid;
            else hi = mid - 1;
        }
        const int64_t bk = lo;
        const uint64_t ub = uoff[bk];
        const int64_t sub = u - (int64_t)(uint32_t)ub;
        const int64_t ns = (int64_t)(uint32_t)uoff[bk + 1] - (int64_t)(uint32_t)ub;
        const int64_t s = start[bk] + sub * kUnitItems;
        const int64_t e = s + kUnitItems < start[bk + 1] ? s + kUnitItems : start[bk + 1];
        for (int q = lane; q < 2 * rows; q += 64) acc[q] = 0.0f;
        wave_lds_sync();
        reduce_range(keys, vals, s, e, B, acc);
        if (ns == 1) {
            const int64_t row0 = bk << B;
            for (int q = lane; q < rows; q += 64) {
                const int64_t row = row0 + q;
                if (row < (int64_t)n_entries)
                    *reinterpret_cast<float2*>(out + 2 * row) =
                        make_float2(acc[2 * q], acc[2 * q + 1]);
            }
        } else {
            float* dst = partial + ((int64_t)(ub >> 32) + sub) * (2 * rows);
            for (int q = lane; q < 2 * rows; q += 64) dst[q] = acc[q];
        }
        wave_lds_sync();
    }
}

// Multi-unit buckets: each row is the sum of its units' partials in unit
// order (one wave per bucket, grid-stride).
__global__ void __launch_bounds__(256) k_bucket_combine(const uint64_t* __restrict__ uoff,
                                                        int64_t n_buckets, int B,
                                                        uint32_t n_entries, float* __restrict__ out,
                                                        const float* __restrict__ partial) {
    const int lane = threadIdx.x & 63;
    const int rows = 1 << B;
    for (int64_t bk = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
         bk < n_buckets; bk += (int64_t)gridDim.x * (blockDim.x >> 6)) {
        const uint64_t ub = uoff[bk];
        const int64_t ns = (int64_t)(uint32_t)uoff[bk + 1] - (int64_t)(uint32_t)ub;
        if (ns < 2) continue;
        const float* src = partial + (int64_t)(ub >> 32) * (2 * rows);
        for (int q = lane; q < rows; q += 64) {
            const int64_t row = (bk << B) + q;
            if (row >= (int64_t)n_entries) continue;
            float a = 0.0f, b = 0.0f;
            for (int64_t j = 0; j < ns; ++j) {
                a += src[j * 2 * rows + 2 * q];
                b += src[j * 2 * rows + 2 * q + 1];
            }
            *reinterpret_cast<float2*>(out + 2 * row) = make_float2(a, b);
        }
    }
}

// ---- paged form: kernels ----
__device__ __forceinline__ int level_digits(const TableLevels& t, int l) {
    return (int)((t.offset[l + 1] - t.offset[l] + (uint32_t)kRows - 1u) >> kRowBits);
}

// One wave, lane = level: page bounds (never past the arrays), slices and work
// units.
__global__ void k_page_plan(TableLevels t, const uint64_t* __restrict__ scan, int64_t units,
                            int active, int64_t per_level, int64_t capacity,
                            PagePlan* __restrict__ plan) {
    const int l = threadIdx.x;
    const bool on = l < t.L;
    auto first_page = [&](int q) -> int64_t {
        if (q > active) q = active;
        const int64_t p = scan ? (int64_t)(scan[q * units] >> 40) : q * per_level;
        return p < capacity ? p : capacity;
    };
    const int64_t p = on ? first_page(l) : 0, n = on ? (first_page(l + 1) - p) * kPage : 0;
    const int64_t total = first_page(t.L) * kPage;
    int64_t unit = total / 1024;
    unit = unit < kUnitLeast ? kUnitLeast : (unit > kUnitMost ? kUnitMost : unit);
    const int D = on ? level_digits(t, l) : 0;
    int64_t S = on ? (n + D * unit - 1) / (D * unit) : 0;
    if (on && S < 1) S = 1;
    const uint32_t all = (uint32_t)(D * S);
    const uint32_t slots = S > 1 ? all : 0u;
    const uint32_t rows = S > 1 ? t.offset[l + 1] - t.offset[l] : 0u;   // combined afterwards
    const uint32_t us = wave_scan(all), ss = wave_scan(slots), rs = wave_scan(rows);
    const uint32_t sum = __shfl(us, 63, 64);
    if (on) {
        plan->page_base[l] = (int32_t)p;
        // finest level first: its buckets hold the most pairs
        plan->unit_base[l] = (int32_t)(sum - us);
        plan->slices[l] = (int32_t)S;
        plan->slot_base[l] = (int32_t)(ss - slots);
        plan->row_base[l] = (int32_t)(rs - rows);
        if (l == t.L - 1) {
            plan->page_base[l + 1] = (int32_t)(p + n / kPage);
            plan->row_base[l + 1] = (int32_t)rs;
        }
        if (l == 0) plan->unit_base[t.L] = (int32_t)sum;
    }
}

// Runs of one bucket in pages [p0, p1) of a level: a wave takes every 16th
// page.  Its lanes look 64 runs up at once; each run is read by the whole
// wave, 64 pairs a load, eight runs' loads in flight together.  body.load(base,
// i): pair base + i of the arrays (base is the same for the wave);
// body.use(payload).  Returns the pairs of the runs that this lane looked up.
struct RunSpan {
    const uint16_t* run_start;   // the level's first page, at the bucket
    int64_t first;               // the level's first pair
    int p0, p1;
};

template <class Body>
__device__ __forceinline__ uint32_t for_runs(const RunSpan& s, const Body& body) {
    constexpr int kU = 8;
    const uint32_t lane = threadIdx.x & 63u;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint32_t total = 0;
    for (int b = s.p0 + wave; b < s.p1; b += 16 * 64) {
        const int mine = b + 16 * (int)lane;
        uint32_t both = 0;   // two neighbouring 16-bit entries: start, end
        if (mine < s.p1) __builtin_memcpy(&both, s.run_start + (int64_t)mine * kRunStride, 4);
        total += (both >> 16) - (both & 0xffffu);
        const int runs = (s.p1 - b + 15) / 16 < 64 ? (s.p1 - b + 15) / 16 : 64;
        for (int q = 0; q < runs; q += kU) {
            const int64_t base0 = s.first + (int64_t)(b + 16 * q) * kPage;
            uint32_t st[kU], len[kU];
            typename Body::Payload v[kU];
            bool longer = false;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)both, (q + u) & 63);
                st[u] = d & 0xffffu;
                len[u] = (d >> 16) - st[u];
                longer = longer || len[u] > 64u;
                if (lane < len[u]) v[u] = body.load(base0 + (int64_t)(u * 16 * kPage) + st[u], lane);
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (lane < len[u]) body.use(v[u]);
            if (!longer) continue;
#pragma unroll 1
            for (int u = 0; u < kU; ++u) {
                const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)both, (q + u) & 63);
                const uint32_t n = (d >> 16) - (d & 0xffffu);
                const int64_t base = base0 + (int64_t)(u * 16 * kPage) + (d & 0xffffu);
                for (uint32_t j = 64; j < n; j += 256) {
                    typename Body::Payload w[4];
#pragma unroll
                    for (uint32_t c = 0; c < 4; ++c)
                        if (j + 64 * c + lane < n) w[c] = body.load(base + j, 64 * c + lane);
#pragma unroll
                    for (uint32_t c = 0; c < 4; ++c)
                        if (j + 64 * c + lane < n) body.use(w[c]);
                }
            }
        }
    }
    return total;
}

// The rows' largest exponents.
struct RunMax {
    using Payload = uint32_t;
    const uint32_t* keys;
    uint32_t* mx;
    __device__ __forceinline__ uint32_t load(int64_t base, uint32_t i) const {
        return (keys + base)[i];
    }
    __device__ __forceinline__ void use(uint32_t w) const {
        const uint32_t row = w & (uint32_t)(kRows - 1);
        atomicMax(&mx[row], w >> kRowBits & 255u);
        atomicMax(&mx[kRows + row], w >> (kRowBits + 8));
    }
};

// v as a multiple of its row's grid, 2^(e - 126 - Q) with e the row's largest
// exponent: the low bits of v + c, c = 1.5 * 2^52 grid steps, less c's.
// ck = (897 + 52 - Q) << 20 | 0x80000: c's high word is (e << 20) + ck.
__device__ __forceinline__ unsigned long long grid_steps(float v, uint32_t e, uint32_t ck) {
    const uint32_t ch = (e << 20) + ck;
    const double x = (double)v + __hiloint2double((int)ch, 0);
    return (unsigned long long)((uint32_t)__double2hiint(x) - ch) << 32 |
           (uint32_t)__double2loint(x);
}

// A value added to a row with an infinity or NaN: flags (1 NaN, 2 +inf,
// 4 -inf) in place of the sum.
__device__ __forceinline__ void add_special(float v, unsigned long long* acc) {
    const uint32_t b = __float_as_uint(v);
    if ((b & 0x7f800000u) != 0x7f800000u) return;
    const uint32_t f = (b & 0x7fffffu) ? 1u : ((b >> 31) ? 4u : 2u);
    atomicOr(reinterpret_cast<uint32_t*>(acc), f);
}

// The values added up; kSpecial: some row of the bucket holds an infinity or
// NaN.
template <class VT, bool kSpecial>
struct RunAdd {
    struct Payload {
        uint32_t w;
        VT v;
    };
    const uint32_t* keys;
    const VT* vals;
    const uint16_t* ex;
    unsigned long long* acc;
    uint32_t ck;
    __device__ __forceinline__ Payload load(int64_t base, uint32_t i) const {
        return Payload{(keys + base)[i], (vals + base)[i]};
    }
    __device__ __forceinline__ void use(const Payload& p) const {
        const float2 v = pair_value(p.v);
        const uint32_t row = p.w & (uint32_t)(kRows - 1);
        const uint32_t e = ex[row], e0 = e & 255u, e1 = e >> 8;
        if (kSpecial && e0 == 255u) add_special(v.x, &acc[row]);
        else atomicAdd(&acc[row], grid_steps(v.x, e0, ck));
        if (kSpecial && e1 == 255u) add_special(v.y, &acc[kRows + row]);
        else atomicAdd(&acc[kRows + row], grid_steps(v.y, e1, ck));
    }
};

// The sum of a row: its steps times the grid.
__device__ __forceinline__ double row_sum(unsigned long long a, uint32_t e, int Q) {
    if (e == 255u) {
        const uint32_t f = (uint32_t)a;
        const double inf = __hiloint2double(0x7ff00000, 0);
        return f == 2u ? inf : (f == 4u ? -inf : __hiloint2double(0x7ff80000, 0));
    }
    return ldexp((double)(long long)a, (int)e - 126 - Q);
}

// One block per work unit: a bucket of 8192 rows, or a slice of its level's
// pages.  Two passes over the bucket's runs: the largest exponent of each
// row (LDS max over the key words), then the values, as whole
// numbers of their row's grid, added into 64-bit integers in LDS.  With at
// most 2^b pairs in the unit, the grid is 2^-Q of the row's largest binade,
// Q = min(50, 61 - b), so the integer sums cannot overflow and are exact in
// any order: no sort, no barrier between the additions, and the same bits on
// every run.  A value's rounding to the grid (2^-45 of the row's largest at
// 10^5 pairs a unit; none for values within 2^-21 of it) is far below that
// of a float sum.
// 1024 threads and 144 KB of LDS (the first pass's maxima lie where the sums
// go, and are packed to 16 bits a row before the second): one block a CU.
template <class VT>
__global__ void __launch_bounds__(1024) k_page_reduce(TableLevels t,
                                                      const PagePlan* __restrict__ plan,
                                                      const uint32_t* __restrict__ keys,
                                                      const VT* __restrict__ vals,
                                                      const uint16_t* __restrict__ run_start,
                                                      float* __restrict__ out,
                                                      double2* __restrict__ partial) {
    __shared__ unsigned long long acc[2 * kRows];
    __shared__ uint16_t ex[kRows];
    __shared__ uint32_t pairs;
    uint32_t* mx = reinterpret_cast<uint32_t*>(acc);
    const int tid = (int)threadIdx.x;
    // blocks b, b + 8, ... share an XCD: 32 neighbouring units at a time, whose
    // runs share cache lines
    const int bx = (int)blockIdx.x & 7, by = (int)blockIdx.x >> 3;
    const int u = ((by >> 5) * 8 + bx) * 32 + (by & 31);
    if (u >= plan->unit_base[t.L]) return;
    int l = t.L - 1;
    while (l > 0 && u >= plan->unit_base[l - 1]) --l;
    const int D = level_digits(t, l), S = plan->slices[l];
    const int v = u - plan->unit_base[l];
    const int slice = v / D, d = v - slice * D;
    const int pb = plan->page_base[l], np = plan->page_base[l + 1] - pb;
    RunSpan s;
    s.run_start = run_start + (int64_t)pb * kRunStride + d;
    s.first = (int64_t)pb * kPage;
    s.p0 = (int)((int64_t)np * slice / S);
    s.p1 = (int)((int64_t)np * (slice + 1) / S);
    for (int q = tid; q < 2 * kRows; q += 1024) mx[q] = 0u;
    if (tid == 0) pairs = 0u;
    __syncthreads();
    const uint32_t mine = wave_scan(for_runs(s, RunMax{keys, mx}));
    if ((tid & 63) == 63) atomicAdd(&pairs, mine);
    __syncthreads();
    bool special = false;
    for (int q = tid; q < kRows; q += 1024) {
        const uint32_t e0 = mx[q], e1 = mx[kRows + q];
        special = special || e0 == 255u || e1 == 255u;
        ex[q] = (uint16_t)(e0 | e1 << 8);
    }
    special = __syncthreads_or(special) != 0;
    for (int q = tid; q < 2 * kRows; q += 1024) acc[q] = 0ull;
    const int b = pairs > 1u ? 32 - __clz((int)(pairs - 1u)) : 0;
    const int Q = 61 - b < 50 ? 61 - b : 50;
    const uint32_t ck = (uint32_t)(897 + 52 - Q) << 20 | 0x80000u;
    __syncthreads();
    if (special) for_runs(s, RunAdd<VT, true>{keys, vals, ex, acc, ck});
    else for_runs(s, RunAdd<VT, false>{keys, vals, ex, acc, ck});
    __syncthreads();
    const uint32_t rows = t.offset[l + 1] - t.offset[l];
    double2* dst = partial + ((int64_t)(plan->slot_base[l] + d * S + slice) << kRowBits);
#pragma unroll
    for (int r = 0; r < kRows / 1024; ++r) {
        const int q = tid + 1024 * r;
        const uint32_t e = ex[q];
        const double x = row_sum(acc[q], e & 255u, Q), y = row_sum(acc[kRows + q], e >> 8, Q);
        const uint32_t row = (uint32_t)d * kRows + q;
        if (S > 1) dst[q] = make_double2(x, y);
        else if (row < rows)
            *reinterpret_cast<float2*>(out + 2 * ((int64_t)t.offset[l] + row)) =
                make_float2((float)x, (float)y);
    }
}

// Sliced levels: each row is the sum of its slices' partials in order.
__global__ void __launch_bounds__(256) k_page_combine(TableLevels t,
                                                      const PagePlan* __restrict__ plan,
                                                      const double2* __restrict__ partial,
                                                      float* __restrict__ out) {
    const uint32_t all = (uint32_t)plan->row_base[t.L];
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < all; i += gridDim.x * 256u) {
        int l = 0;
        while (i >= (uint32_t)plan->row_base[l + 1]) ++l;
        const uint32_t q = i - (uint32_t)plan->row_base[l];
        const int S = plan->slices[l];
        const double2* src = partial +
                             ((int64_t)(plan->slot_base[l] + (int)(q >> kRowBits) * S) << kRowBits) +
                             (q & (uint32_t)(kRows - 1));
        double a = 0.0, b = 0.0;
#pragma unroll 4
        for (int j = 0; j < S; ++j) {
            const double2 p = src[(int64_t)j << kRowBits];
            a += p.x;
            b += p.y;
        }
        *reinterpret_cast<float2*>(out + 2 * ((int64_t)t.offset[l] + q)) =
            make_float2((float)a, (float)b);
    }
}

void table_pages_carve(WsCarver& c, int64_t pages, bool half_vals, TablePages* out) {
    TablePages w{};
    w.pages = pages;
    w.half_vals = half_vals;
    w.keys = c.take<uint32_t>((size_t)pages * kPage);
    w.vals = c.take<char>((size_t)pages * kPage * (half_vals ? 4 : 8));
    w.run_start = c.take<uint16_t>((size_t)pages * kRunStride + 2);
    w.partial = c.take<double2>((size_t)slot_bound(pages * kPage) << kRowBits);
    w.plan = c.take<PagePlan>(1);
    *out = w;
}

int table_pages_plan(TablePages& w, const am_grid_desc* g, const uint64_t* scan, int64_t units,
                     int active, int64_t per_level, hipStream_t s) {
    hipLaunchKernelGGL(k_page_plan, dim3(1), dim3(64), 0, s, table_levels(g), scan, units, active,
                       per_level, w.pages, w.plan);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <class VT>
static int run_pages(TablePages& w, const am_grid_desc* g, float* dtable, hipStream_t s) {
    const TableLevels t = table_levels(g);
    KernelTimer kt_("seg_reduce", s);
    // units <= buckets + pairs / unit pairs (both unit sizes of k_page_plan)
    const int64_t m = w.pages * kPage, least = m / kUnitLeast, most = m / kUnitMost;
    const int64_t units = table_digits(g) + (least < 1024 ? least : (most > 1024 ? most : 1024)) + 2;
    const unsigned grid = (unsigned)(ceil_div(units, 256) * 256);   // whole groups of 8 x 32
    hipLaunchKernelGGL((k_page_reduce<VT>), dim3(grid), dim3(1024), 0, s, t, w.plan, w.keys,
                       reinterpret_cast<const VT*>(w.vals), w.run_start, dtable, w.partial);
    AM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_page_combine, dim3(2048), dim3(256), 0, s, t, w.plan, w.partial, dtable);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

int table_pages_run(TablePages& w, const am_grid_desc* g, float* dtable, hipStream_t s) {
    return w.half_vals ? run_pages<uint32_t>(w, g, dtable, s) : run_pages<uint2>(w, g, dtable, s);
}

template <class VT>
static int run_bucketed(TableReduceWs& w, uint32_t n_entries, float* dtable, hipStream_t s) {
    uint32_t* ks = w.keys[0];
    VT* vs = reinterpret_cast<VT*>(w.vals[0]);
    if (w.m > 0) {
        size_t sb = w.sort_bytes;
        hipError_t e;
        {
            KernelTimer kt_("radix_sort", s);
            e = sort_pairs<VT>(w.sort_tmp, sb, w, &ks, &vs, s);
        }
        if (e != hipSuccess) {
            set_error("radix sort failed: %s", hipGetErrorString(e));
            return AM_ERR_HIP;
        }
    }
    KernelTimer kt_("seg_reduce", s);
    const unsigned gb = (unsigned)ceil_div(w.n_buckets + 1, 256);
    hipLaunchKernelGGL(k_bucket_bounds, dim3(gb), dim3(256), 0, s, ks, w.m, w.begin_bit,
                       w.n_buckets, w.bucket_start);
    AM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_bucket_units, dim3(gb), dim3(256), 0, s, w.bucket_start, w.n_buckets,
                       w.units);
    AM_LAUNCH_CHECK();
    size_t scb = w.scan_bytes;
    hipError_t e = rocprim::exclusive_scan(w.scan_tmp, scb, w.units, w.unit_off, (uint64_t)0,
                                           (size_t)w.n_buckets + 1, rocprim::plus<uint64_t>(), s,
                                           false);
    if (e != hipSuccess) {
        set_error("bucket unit scan failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    // units <= n_buckets + m / kUnitItems + 1; the kernel reads the total
    const int64_t max_units = w.n_buckets + w.m / kUnitItems + 1;
    const int64_t want = ceil_div(max_units, kBucketWaves);
    const unsigned grid = (unsigned)(want < 8192 ? want : 8192);
    hipLaunchKernelGGL((k_bucket_reduce<VT>), dim3(grid), dim3(64 * kBucketWaves), 0, s, ks, vs,
                       w.bucket_start, w.unit_off, w.n_buckets, w.begin_bit, n_entries, dtable,
                       w.partial);
    AM_LAUNCH_CHECK();
    const int64_t cw = ceil_div(w.n_buckets, 4);
    hipLaunchKernelGGL(k_bucket_combine, dim3((unsigned)(cw < 4096 ? cw : 4096)), dim3(256), 0, s,
                       w.unit_off, w.n_buckets, w.begin_bit, n_entries, dtable, w.partial);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

int fill_f32(float* p, int64_t n, float v, hipStream_t s) {
    if (n <= 0) return AM_OK;
    int blocks = (int)(ceil_div(n, 256) < 8192 ? ceil_div(n, 256) : 8192);
    hipLaunchKernelGGL(k_fill_f32, dim3(blocks), dim3(256), 0, s, p, n, v);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

template <int F, class VT>
static int run_f(TableReduceWs& w, uint32_t n_entries, float* dtable, hipStream_t s) {
    if (int rc = fill_f32(dtable, (int64_t)n_entries * F, 0.0f, s)) return rc;
    if (w.m == 0) return AM_OK;
    uint32_t* ks = nullptr;
    VT* vs = nullptr;
    size_t sb = w.sort_bytes;
    hipError_t e;
    {
        KernelTimer kt_("radix_sort", s);
        e = sort_pairs<VT>(w.sort_tmp, sb, w, &ks, &vs, s);
    }
    if (e != hipSuccess) {
        set_error("radix sort failed: %s", hipGetErrorString(e));
        return AM_ERR_HIP;
    }
    const int64_t nc = ceil_div(w.m, kSegChunk);
    const int gb = (int)ceil_div(nc, 256);
    {
        KernelTimer kt_("seg_reduce", s);
        constexpr int T = SegCfg<F>::threads;
        hipLaunchKernelGGL((k_seg_a<F, VT>), dim3((unsigned)ceil_div(nc, T)), dim3(T), 0, s, ks, vs, w.m,
                           n_entries, dtable, w.lead, w.tail, w.lead_full, w.tail_open);
    }
    AM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_seg_b<F>, dim3(gb), dim3(256), 0, s, ks, w.m, n_entries, dtable, w.lead,
                       w.tail, w.lead_full, w.tail_open);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

int table_reduce_run(TableReduceWs& w, const am_grid_desc* g, float* dtable,
                     hipStream_t stream) {
    const int F = g->n_features;
    const uint32_t n_entries = g->n_entries;
    if (F == 2 && w.n_buckets > 0) {
        if (w.begin_bit > kMaxBucketBits) {
            set_error("bucket bits %d above %d", w.begin_bit, kMaxBucketBits);
            return AM_ERR_INTERNAL;
        }
        return w.half_vals ? run_bucketed<ValsH<2>>(w, n_entries, dtable, stream)
                           : run_bucketed<Vals<2>>(w, n_entries, dtable, stream);
    }
    if (w.half_vals) {
        if (F == 2) return run_f<2, ValsH<2>>(w, n_entries, dtable, stream);
        set_error("fp16 gradient pairs need n_features = 2 (got %d)", F);
        return AM_ERR_UNSUPPORTED;
    }
    switch (F) {
        case 1: return run_f<1, Vals<1>>(w, n_entries, dtable, stream);
        case 2: return run_f<2, Vals<2>>(w, n_entries, dtable, stream);
        case 4: return run_f<4, Vals<4>>(w, n_entries, dtable, stream);
        case 8: return run_f<8, Vals<8>>(w, n_entries, dtable, stream);
        default: set_error("unsupported n_features %d", F); return AM_ERR_UNSUPPORTED;
    }
}

}  // namespace am
