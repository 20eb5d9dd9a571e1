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
// Pairs of a work unit: a bucket of more than half as many again is cut into
// slices of about this many, a 1216th of all pairs between the two bounds: with
// what the buckets round up, just under five rounds of 256 blocks.  Fewer, longer
// units end raggedly; one more than a round starts another; more units write
// and merge more partial sums.  Reduce and merge with 768 / 960 / 1024 / 1216 /
// 1440 / 2048 units: 940 k samples, 16 levels 1930 / 1925 / 1911 / 1827 / 1760 /
// 1776 us; 480 k, 4 levels 576 / 584 / 667 / 586 / 659 / 774; 240 k, 16 levels
// of 2^19 rows 438 / 469 / - / 420 / 441 / -.  With 16384 / 32768 / 49152 /
// 65536 pairs at least: 65 k samples, 8 levels 133 / 96 / 74 / 94 us; the
// background's 29 M pairs - / 244 / 242 / 259; 65 k samples, 16 levels - / 164 /
// 186 / 187.
constexpr int64_t kUnitMost = 1 << 19;
constexpr int64_t kUnitLeast = 49152;
constexpr int64_t kUnits = 1216;
__host__ __device__ inline int64_t unit_pairs(int64_t total) {
    const int64_t u = total / kUnits;
    return u < kUnitLeast ? kUnitLeast : (u > kUnitMost ? kUnitMost : u);
}

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
    for (int l = 0; l < g->n_levels; ++l) {
        t.bucket[l] = t.n_buckets;
        t.n_buckets += (int32_t)ceil_div(g->size[l], kRows);
    }
    return t;
}

// At most n / U for the unit U of any number n of pairs up to m.
static int64_t units_of(int64_t m) {
    const int64_t a = m / kUnitLeast, b = m / kUnitMost;
    return (a < kUnits ? a : (b > kUnits ? b : kUnits)) + 1;
}
// A sliced bucket of n > 1.5 U pairs has S = ceil(n / U) <= 1.5 n / U slices.
static int64_t slot_bound(int64_t m) { return 3 * units_of(m) / 2 + 1; }

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

__device__ __forceinline__ int64_t first_page(const PageSource& src, int level) {
    const int q = level < src.active ? level : src.active;
    const int64_t p = src.scan ? (int64_t)(src.scan[q * src.units] >> 40) : q * src.per_level;
    return p < src.capacity ? p : src.capacity;
}

constexpr int kMostChunks = 16;

// Pairs of each bucket in a part of its level's pages, from the run tables.
// Block (part, level); 1024 threads: the buckets, four pages at a time.
__global__ void __launch_bounds__(1024) k_bucket_pairs(TableLevels t, PageSource src,
                                                       const uint16_t* __restrict__ run_start,
                                                       uint32_t* __restrict__ pairs) {
    __shared__ uint32_t part[4][kMaxDigits];
    const int l = (int)blockIdx.y, d = (int)threadIdx.x & (kMaxDigits - 1), q = (int)threadIdx.x >> 8;
    const int64_t p0 = first_page(src, l), np = first_page(src, l + 1) - p0;
    const int64_t a = p0 + np * blockIdx.x / gridDim.x, b = p0 + np * (blockIdx.x + 1) / gridDim.x;
    const int D = level_digits(t, l);
    uint32_t sum = 0;
    if (d < D) {
#pragma unroll 8
        for (int64_t p = a + q; p < b; p += 4) {
            const uint16_t* rs = run_start + p * kRunStride + d;
            sum += (uint32_t)rs[1] - (uint32_t)rs[0];
        }
    }
    part[q][d] = sum;
    __syncthreads();
    if (q == 0 && d < D)
        pairs[(int64_t)blockIdx.x * t.n_buckets + t.bucket[l] + d] =
            (part[0][d] + part[1][d]) + (part[2][d] + part[3][d]);
}

// Exclusive sum over the block's 1024 threads, and the total.
__device__ __forceinline__ uint64_t block_scan(uint64_t v, uint64_t* wave_sum, uint64_t* total) {
    const int tid = (int)threadIdx.x;
    uint64_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up((unsigned long long)incl, d, 64);
        if ((tid & 63) >= d) incl += o;
    }
    if ((tid & 63) == 63) wave_sum[tid >> 6] = incl;
    __syncthreads();
    uint64_t at = incl - v, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        if (w < tid >> 6) at += wave_sum[w];
        all += wave_sum[w];
    }
    __syncthreads();
    *total = all;
    return at;
}

// The work units: each bucket's pairs cut into slices by its own load, so that
// samples that crowd in few cells are spread over the chip like any others.
// With slices by the level's mean load the fullest bucket of a fine level was
// one block's: 940 k samples within 0.002 of a point, 2^21 rows a level, reduce
// 7.6 -> 3.3 ms, within 0.1: 2.76 -> 2.52; 2 M points of the stand-alone grid
// within 0.4 % of the box 29.5 -> 5.3 ms.  Spread samples pay 5 to 10 us for
// the counts (20 k samples: 87 -> 91 us in all).  Counts and units in one launch
// were no faster: with the units cut by the last of the counting blocks its
// fences write the emission's dirty lines back (27 to 54 us), and with a range
// of units for each level every block pays for finding its unit (20 k samples,
// reduce 72 -> 77 us) or the XCDs for the ranges' gaps (29 M pairs 231 -> 245).
// Buckets without pairs have no unit; the merge writes their zeros.
__global__ void __launch_bounds__(1024) k_page_plan(TableLevels t, PageSource src,
                                                    const uint16_t* __restrict__ run_start,
                                                    const uint32_t* __restrict__ pairs, int chunks,
                                                    PagePlan* __restrict__ plan,
                                                    PageUnit* __restrict__ units,
                                                    PageUnit* __restrict__ merges) {
    constexpr int kMost = AM_MAX_LEVELS * kMaxDigits;
    __shared__ uint64_t n[kMost + 1];   // pairs, then the scan
    __shared__ uint64_t wave_sum[16];
    const int tid = (int)threadIdx.x, each = (t.n_buckets + 1023) / 1024;
    // four waves to a level, whose parameters are scalars
    const int quarter = __builtin_amdgcn_readfirstlane(tid >> 8), d = tid & (kMaxDigits - 1);
    uint64_t sum = 0, total;
    if (chunks > 0) {
        for (int i = tid; i < t.n_buckets; i += 1024) {
            uint64_t v = 0;
#pragma unroll
            for (int c = 0; c < kMostChunks; ++c)
                v += c < chunks ? pairs[(int64_t)c * t.n_buckets + i] : 0u;
            n[i] = v;
            sum += v;
        }
    } else {   // few pages: from the run tables themselves
        for (int l = quarter; l < t.L; l += 4) {
            if (d >= level_digits(t, l)) continue;
            const int64_t p1 = first_page(src, l + 1);
            uint64_t v = 0;
            for (int64_t p = first_page(src, l); p < p1; ++p) {
                const uint16_t* rs = run_start + p * kRunStride + d;
                v += (uint32_t)rs[1] - (uint32_t)rs[0];
            }
            n[t.bucket[l] + d] = v;
            sum += v;
        }
    }
    block_scan(sum, wave_sum, &total);
    const uint64_t U = (uint64_t)unit_pairs((int64_t)total);
    // units | partial slots << 24 | merges << 48
    auto counts = [&](uint64_t m) -> uint64_t {
        if (m != 0u && m <= U + U / 2u) return 1u;
        const uint64_t S = m >> 32 ? (m + U - 1u) / U
                                   : (uint32_t)m / (uint32_t)U + ((uint32_t)m % (uint32_t)U != 0u);
        return S | S << 24 | 1ull << 48;
    };
    const int i0 = tid * each < t.n_buckets ? tid * each : t.n_buckets;
    const int i1 = i0 + each < t.n_buckets ? i0 + each : t.n_buckets;
    uint64_t mine = 0;
    for (int i = i0; i < i1; ++i) mine += n[i] = counts(n[i]);
    uint64_t at = block_scan(mine, wave_sum, &total);
    for (int i = i0; i < i1; ++i) {
        const uint64_t c = n[i];
        n[i] = at;
        at += c;
    }
    if (tid == 0) {
        n[t.n_buckets] = total;
        plan->n_units = (int32_t)(total & 0xffffffu);
        plan->n_merges = (int32_t)(total >> 48);
    }
    __syncthreads();
    for (int l = quarter; l < t.L; l += 4) {
        if (d >= level_digits(t, l)) continue;
        const uint64_t a = n[t.bucket[l] + d], b = n[t.bucket[l] + d + 1];
        const int64_t p0 = first_page(src, l);
        const int pages = (int)(first_page(src, l + 1) - p0), first = (int)(a & 0xffffffu);
        const uint32_t left = t.offset[l + 1] - t.offset[l] - (uint32_t)d * kRows;
        PageUnit w;
        w.slices = (int)(b & 0xffffffu) - first;
        w.bucket = d;
        w.row = t.offset[l] + (uint32_t)d * kRows;
        w.rows = left < (uint32_t)kRows ? left : (uint32_t)kRows;
        w.page = p0;
        w.slot = (int)(a >> 24 & 0xffffffu);
        w.runs = 0;
        if (a >> 48 != b >> 48) merges[a >> 48] = w;
        for (int q = 0; q < w.slices; ++q) {   // every slices-th page from the q-th on
            w.runs = (pages - q + w.slices - 1) / w.slices;
            units[first + q] = w;
            ++w.page;
            ++w.slot;
        }
    }
}

// Runs of one bucket in every step-th page of a level: a wave takes every 16th
// of them.  Its lanes look 64 runs up at once; each run is read by the whole
// wave, 64 pairs a load, eight runs' loads in flight together.  body.load(base,
// i): pair base + i of the arrays (base is the same for the wave);
// body.use(payload).  Returns the pairs of the runs that this lane looked up.
struct RunSpan {
    const uint16_t* run_start;   // the first page, at the bucket
    int64_t first;               // the first page's first pair
    int runs, step;              // pages, and from one to the next
};

template <class Body>
__device__ __forceinline__ uint32_t for_runs(const RunSpan& s, const Body& body) {
    constexpr int kU = 8;
    const uint32_t lane = threadIdx.x & 63u;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int64_t apart = (int64_t)s.step * (16 * kPage);   // a wave's runs
    uint32_t total = 0;
    for (int b = wave; b < s.runs; b += 16 * 64) {
        const int mine = b + 16 * (int)lane;
        uint32_t both = 0;   // two neighbouring 16-bit entries: start, end
        if (mine < s.runs)
            __builtin_memcpy(&both, s.run_start + (int64_t)mine * s.step * kRunStride, 4);
        total += (both >> 16) - (both & 0xffffu);
        const int runs = (s.runs - b + 15) / 16 < 64 ? (s.runs - b + 15) / 16 : 64;
        for (int q = 0; q < runs; q += kU) {
            int64_t base0 = s.first + (int64_t)b * s.step * kPage + q * apart;
            uint32_t st[kU], len[kU];
            typename Body::Payload v[kU];
            bool longer = false;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)both, (q + u) & 63);
                st[u] = d & 0xffffu;
                len[u] = (d >> 16) - st[u];
                longer = longer || len[u] > 64u;
                if (lane < len[u]) v[u] = body.load(base0 + st[u], lane);
                base0 += apart;
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (lane < len[u]) body.use(v[u]);
            if (!longer) continue;
            base0 -= kU * apart;
#pragma unroll 1
            for (int u = 0; u < kU; ++u, base0 += apart) {
                const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)both, (q + u) & 63);
                const uint32_t n = (d >> 16) - (d & 0xffffu);
                const int64_t base = base0 + (d & 0xffffu);
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

// One block per work unit: a bucket of 8192 rows, or every S-th page's part of
// it.  Two passes over the bucket's runs: the largest exponent of each
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
__global__ void __launch_bounds__(1024) k_page_reduce(const PagePlan* __restrict__ plan,
                                                      const PageUnit* __restrict__ units,
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
    if (u >= plan->n_units) return;
    const PageUnit w = units[u];
    RunSpan s;
    s.run_start = run_start + w.page * kRunStride + w.bucket;
    s.first = w.page * kPage;
    s.step = w.slices;
    s.runs = w.runs;
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
    double2* dst = partial + ((int64_t)w.slot << kRowBits);
    float2* row = reinterpret_cast<float2*>(out) + w.row;
#pragma unroll
    for (int r = 0; r < kRows / 1024; ++r) {
        const int q = tid + 1024 * r;
        if ((uint32_t)q >= w.rows) continue;
        const uint32_t e = ex[q];
        const double x = row_sum(acc[q], e & 255u, Q), y = row_sum(acc[kRows + q], e >> 8, Q);
        if (w.slices > 1) dst[q] = make_double2(x, y);
        else row[q] = make_float2((float)x, (float)y);
    }
}

// Buckets of several slices: each row is the sum of its slices' partials, in
// one order for a number of slices; buckets without pairs: zeros.  A block
// takes 512 rows; from 8 slices on, 64 rows at a time by four waves, a quarter
// of the slices each (a single level of 72 rows with 16 M pairs, where hundreds
// of slices meet: backward 596 -> 383 us).
__global__ void __launch_bounds__(256) k_page_merge(const PagePlan* __restrict__ plan,
                                                    const PageUnit* __restrict__ merges,
                                                    const double2* __restrict__ partial,
                                                    float* __restrict__ out) {
    constexpr int kPart = 512;
    __shared__ double2 sums[4][64];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int all = plan->n_merges * (kRows / kPart);
    for (int e = (int)blockIdx.x; e < all; e += (int)gridDim.x) {
        const PageUnit m = merges[e / (kRows / kPart)];
        const int slices = m.slices, q0 = e % (kRows / kPart) * kPart;   // row within the bucket
        const int n = min((int)m.rows - q0, kPart);
        float2* dst = reinterpret_cast<float2*>(out) + m.row + q0;
        const double2* src = partial + ((int64_t)m.slot << kRowBits) + q0;
        if (slices < 8) {
            for (int q = tid; q < n; q += 256) {
                double2 p[7];
#pragma unroll
                for (int j = 0; j < 7; ++j)
                    if (j < slices) p[j] = src[((int64_t)j << kRowBits) + q];
                double2 sum = make_double2(0.0, 0.0);
#pragma unroll
                for (int j = 0; j < 7; ++j)
                    if (j < slices) {
                        sum.x += p[j].x;
                        sum.y += p[j].y;
                    }
                dst[q] = make_float2((float)sum.x, (float)sum.y);
            }
            continue;
        }
        for (int q = 0; q < n; q += 64) {
            double2 sum = make_double2(0.0, 0.0);
            if (q + lane < n)
                for (int j0 = wave; j0 < slices; j0 += 32) {
                    double2 p[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                        if (j0 + 4 * c < slices)
                            p[c] = src[((int64_t)(j0 + 4 * c) << kRowBits) + q + lane];
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                        if (j0 + 4 * c < slices) {
                            sum.x += p[c].x;
                            sum.y += p[c].y;
                        }
                }
            sums[wave][lane] = sum;
            __syncthreads();
            if (wave == 0 && q + lane < n) {
#pragma unroll
                for (int v = 1; v < 4; ++v) {
                    sum.x += sums[v][lane].x;
                    sum.y += sums[v][lane].y;
                }
                dst[q + lane] = make_float2((float)sum.x, (float)sum.y);
            }
            __syncthreads();
        }
    }
}

void table_pages_carve(WsCarver& c, const am_grid_desc* g, int64_t pages, bool half_vals,
                       TablePages* out) {
    const int64_t buckets = table_levels(g).n_buckets;
    TablePages w{};
    w.pages = pages;
    w.half_vals = half_vals;
    w.keys = c.take<uint32_t>((size_t)pages * kPage);
    w.vals = c.take<char>((size_t)pages * kPage * (half_vals ? 4 : 8));
    w.run_start = c.take<uint16_t>((size_t)pages * kRunStride + 2);
    w.partial = c.take<double2>((size_t)slot_bound(pages * kPage) << kRowBits);
    // about 16 pages to a block that counts them; none for a few pages, which
    // the plan counts itself (one launch of 5 us less)
    const int64_t chunks = ceil_div(pages, 16 * (int64_t)g->n_levels);
    w.chunks = (int32_t)(pages <= 4 * (int64_t)g->n_levels
                             ? 0
                             : (chunks > kMostChunks ? kMostChunks : chunks));
    w.pairs = c.take<uint32_t>((size_t)w.chunks * buckets);
    w.plan = c.take<PagePlan>(1);
    w.max_units = buckets + units_of(pages * kPage);   // a bucket's S <= n / U + 1
    w.units = c.take<PageUnit>((size_t)w.max_units);
    w.merges = c.take<PageUnit>((size_t)buckets);
    *out = w;
}

template <class VT>
static int run_pages(TablePages& w, const am_grid_desc* g, const PageSource& src, float* dtable,
                     hipStream_t s) {
    const TableLevels t = table_levels(g);
    KernelTimer kt_("seg_reduce", s);
    if (w.chunks > 0) {
        hipLaunchKernelGGL(k_bucket_pairs, dim3((unsigned)w.chunks, (unsigned)t.L), dim3(1024), 0, s,
                           t, src, w.run_start, w.pairs);
        AM_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_page_plan, dim3(1), dim3(1024), 0, s, t, src, w.run_start, w.pairs,
                       w.chunks, w.plan, w.units, w.merges);
    AM_LAUNCH_CHECK();
    const unsigned grid = (unsigned)(ceil_div(w.max_units, 256) * 256);   // whole groups of 8 x 32
    hipLaunchKernelGGL((k_page_reduce<VT>), dim3(grid), dim3(1024), 0, s, w.plan, w.units, w.keys,
                       reinterpret_cast<const VT*>(w.vals), w.run_start, dtable, w.partial);
    AM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_page_merge, dim3(2048), dim3(256), 0, s, w.plan, w.merges, w.partial,
                       dtable);
    AM_LAUNCH_CHECK();
    return AM_OK;
}

int table_pages_run(TablePages& w, const am_grid_desc* g, const uint64_t* scan, int64_t units,
                    int active, int64_t per_level, float* dtable, hipStream_t s) {
    const PageSource src{scan, units, active, per_level, w.pages};
    return w.half_vals ? run_pages<uint32_t>(w, g, src, dtable, s)
                       : run_pages<uint2>(w, g, src, dtable, s);
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
