// Fused filtered brute-force top-k on the matrix cores (no reference implementation;
// the reference motivates the path only in prose, README.md:265).
//
// For each query q: the k smallest squared L2 distances ||q - x_i||^2 over the
// base vectors i that pass the filter, ascending, ties broken by the smaller id.
//
//   1. tk_enum_count / tk_enum_write: the passing ids of [0, n_base), in
//      ascending order, via GpuRoaringView::contains (any layout, negated too).
//   2. tk_est: distance estimates on the matrix cores, from a two-way f16 split
//      of scaled rows and queries (three f16 MFMA products per fp32 one, with
//      an error no larger than with an fp32 MFMA).  A set of at most `keep` rows
//      gets every estimate written and tk_select picks each query's k from
//      them.  A larger one runs it twice: over a strided sample, from which
//      tk_select bounds each query's k-th distance, and then over every row,
//      where each (query, row) whose estimate could lie at or below that bound
//      is appended to the query's candidate lists.  The second run takes rows
//      and queries about a centre of the query block.
//   3. tk_select: the candidates that can be in the answer get their fp32
//      distance sum((q - x)^2), are ranked by (distance, id), and the first k
//      are written.  Every returned distance is the direct one.
// The estimates only ever gate, with a bound on their error, so the answer does
// not depend on them.  When a query's candidate lists overflow (or the
// estimates are turned off, or its sample says that they would bound little),
// tk_dist and tk_merge answer: per-chunk sorted
// lists under an fp32 MFMA gate, merged by one wave per query.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <type_traits>

#include "cu_roaring/device/roaring_view.hpp"
#include "image.hpp"
#include "internal.hpp"

namespace crimpl {

using cu_roaring::GpuRoaringView;

namespace {

constexpr uint32_t TK_ENUM_IDS = 8192;  // ids per enumeration workgroup
constexpr int TK_ENUM_NT = 256;
constexpr int TK_NT = 512;  // distance kernel: 8 waves
constexpr int TK_WAVES = TK_NT / 64;
constexpr uint32_t TK_QW = 32;                  // queries per wave (MFMA N)
constexpr uint32_t TK_QB = TK_WAVES * TK_QW;    // queries per workgroup
constexpr int TK_ROWS = 64;                     // base rows per tile (two 32-row MFMA blocks)
constexpr uint32_t TK_CB = 512;                 // candidate buffer entries per wave
constexpr uint32_t TK_KMAX = 256;
constexpr uint32_t TK_NOID = 0xFFFFFFFFu;
constexpr int TK_MERGE_NT = 256;
// Bound on |MFMA-expansion distance - fp32 direct distance| per unit of
// |q|^2 + |x|^2 at dim <= 128: about (2*128 + 4) unit roundoffs for the dot
// product, the two norms and the combination, plus the direct sum's own
// 128-term bound, rounded up.
constexpr float TK_GATE_ERR = 4e-5f;
// The MFMA estimate with the (1 - TK_GATE_ERR) scaling is at most the fp32
// distance; adding TK_SEED_ERR (qg + xg) makes it at least the fp32 distance
// (2 E / (1 - E) with E = TK_GATE_ERR, rounded up for the fp32 arithmetic).
constexpr float TK_SEED_ERR = 3.0f * TK_GATE_ERR;
// The same bound for the split estimates (tk_est): 3 x 128 products summed
// at no more than 2^-23 of |q||x| each (4.7e-5 of |q|^2 + |x|^2 with the factor
// 2 of -2 q.x), the split's remainders (2^-22 an element on each side and the
// dropped lo.lo product, 1e-6), the norms and the direct sum (2.3e-5).
constexpr float TK_EST_ERR = 8e-5f;

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Strict order of (distance, id) pairs: the output order.
__device__ __forceinline__ bool tk_less(float ad, uint32_t ai, float bd, uint32_t bi)
{
    return ad < bd || (ad == bd && ai < bi);
}

// Number of entries of the sorted list (d, id)[0, n) that order before (yd, yi).
__device__ __forceinline__ uint32_t tk_lower_bound(const float* d, const uint32_t* id, uint32_t n, float yd,
                                                   uint32_t yi)
{
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tk_less(d[mid], id[mid], yd, yi))
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ uint64_t lanemask_lt() { return (1ull << __lane_id()) - 1ull; }

struct TkArgs {
    const float* base;
    const float* queries;
    const uint32_t* sel;    // passing ids ascending (nullptr: every id of [0, n_base))
    const uint32_t* n_sel;  // device count of sel
    uint64_t n_base;
    uint32_t n_q;
    uint32_t dim;
    uint32_t k;
    uint32_t n_chunks;  // multiple of 8
    uint32_t vec;       // rows are 16-B aligned with dim % 4 == 0
    uint32_t qvec;      // so are the queries
    float* list_d;      // two planes of [n_chunks][n_q][k]: a merge reads one, writes the other
    uint32_t* list_id;  // the same two planes
    size_t plane;       // elements per plane
    uint32_t* list_n;   // [n_chunks][n_q]: list length | (plane holding the list << 31)
    float* gate_at;       // [n_q] the candidates' gate: tau, or -inf for a query that the list path is to answer
    uint32_t* tau_first;  // [n_q] the sample's bound, at which the first candidates are rounded (tau may fall since)
    uint32_t* tau;      // [n_q] bits of the smallest k-th distance any chunk has reached
    uint32_t* tau_m;    // [n_chunks][n_q] bits of each chunk's m_rank-th distance (+inf: fewer entries)
    uint32_t m_rank;    // ceil(2k / n_chunks)
    // The estimate path (gate != 0): sets of at most `keep` rows have every
    // estimate written to pd[q][row], larger ones those of `sample` rows (a
    // power of two, 1 << sample_lg) and then candidates in lists.
    uint32_t gate;
    uint32_t keep;
    uint32_t sample;
    uint32_t sample_lg;
    uint32_t pd_stride;  // row stride of pd: at least keep and sample
    float* pd;           // [whole query blocks][pd_stride] estimates (lower bounds of the fp32 distances)
    uint32_t n_cw;       // candidate lists a query has: one per workgroup of its query block
    uint32_t cap;        // entries of a list
    uint32_t q_rows;     // queries of whole query blocks
    // A query block's centre (tk_centre), where rows and queries are taken about it.
    uint32_t est_qb;     // queries of an estimate workgroup's block
    float* qc;           // [n_q][dim] the queries about their blocks' centres
    float* centre;       // [blocks][128]
    uint32_t* moved;     // [blocks] the centre is not the origin
    uint2* cand;         // [n_cw][n_q][cap] (estimate bits, id)
    uint32_t* cand_n;    // [n_cw][q_rows] candidates found, beyond cap too
    // Up to 64 queries: a query with many candidates is answered by `parts`
    // workgroups, each its part of them; the last one to finish merges.
    uint32_t parts;
    uint64_t* part_key;   // [n_q][parts][k] each part's best, ascending
    uint32_t* part_done;  // [n_q] parts finished
    uint32_t* q_over;    // [n_q] the query's lists overflowed, or would: tk_dist and tk_merge answer it
    uint32_t* qb_over;   // [n_qb] ... any query of the block's
    // What the host launched, from the passing count it knew: with no
    // candidate kernels (or no list path), tk_select answers a set too large
    // (or a query whose lists overflowed) from every passing row.
    uint32_t cand_off;
    uint32_t list_off;
};

// Rows the distance kernels cover, and whether every estimate of them is kept.
__device__ __forceinline__ uint64_t tk_rows(const TkArgs& a) { return a.sel ? static_cast<uint64_t>(*a.n_sel) : a.n_base; }
__device__ __forceinline__ bool tk_small(const TkArgs& a, uint64_t n_rows) { return a.gate != 0 && n_rows <= a.keep; }

// The list path's state when nothing else sets it: every query's bound (tau)
// and each chunk's m_rank-th distance (tau_m) at +inf; thread i of `stride`.
__device__ __forceinline__ void tk_init_from(const TkArgs& a, uint64_t i, uint64_t stride)
{
    if (a.gate) return;
    const uint64_t n = static_cast<uint64_t>(a.n_chunks) * a.n_q;
    for (; i < n; i += stride) {
        a.tau_m[i] = 0x7F800000u;
        if (i < a.n_q) a.tau[i] = 0x7F800000u;
    }
}

// ---- 1. passing ids ---------------------------------------------------------

// A workgroup covers 8192 consecutive ids, a 256-word slice of one key's
// container: the container is looked up once, and thread t takes word t of the
// slice -- from the bitmap, or from the container's image built in LDS for an
// array or run container -- complemented for a negated filter (contains()
// answers `negated` for absent keys) and cut at n_base.
static_assert(TK_ENUM_IDS == 32u * TK_ENUM_NT && 65536u % TK_ENUM_IDS == 0, "one word per thread, one key per block");

__device__ uint32_t tk_enum_word(const GpuRoaringView& v, uint64_t n_base, uint32_t* img, int32_t* cover, int32_t* s_c)
{
    const uint32_t t = threadIdx.x;
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) * TK_ENUM_IDS;
    const uint32_t key = static_cast<uint32_t>(base >> 16);
    if (v.key_index && key <= v.max_key) {
        if (t == 0) {
            const uint16_t e = v.key_index[key];
            *s_c = e == 0xFFFFu ? -1 : static_cast<int32_t>(e);
        }
    } else if (key > v.max_key && v.key_index) {
        if (t == 0) *s_c = -1;
    } else if (t < 64) {
        const uint32_t pos = wave_lower_bound_u16(v.keys, v.n_containers, key);
        if (t == 0) *s_c = (pos < v.n_containers && v.keys[pos] == key) ? static_cast<int32_t>(pos) : -1;
    }
    __syncthreads();
    const int32_t c = *s_c;
    const uint32_t w0 = static_cast<uint32_t>(base & 0xFFFFu) >> 5;  // first word of the slice in the container
    uint32_t word = 0;
    const uint8_t type = c >= 0 ? static_cast<uint8_t>(v.types[c]) : uint8_t(0xFF);  // block-uniform
    if (type == CR_BITMAP) {
        word = reinterpret_cast<const uint32_t*>(v.bitmap_data + v.offsets[c] / 8u)[w0 + t];
    } else if (type == CR_ARRAY || type == CR_RUN) {
        expand_img<TK_ENUM_NT>(type, (type == CR_ARRAY ? v.array_data : v.run_data) + v.offsets[c] / 2u,
                               v.cardinalities[c], img, cover);
        word = img[w0 + t];
    }
    if (v.negated) word = ~word;
    const uint64_t id0 = base + 32u * t;
    if (id0 >= n_base) word = 0;
    else if (n_base - id0 < 32u) word &= (1u << (n_base - id0)) - 1u;
    return word;
}

// Also initialises the call's state (tk_init_from), which saves a launch.
__global__ __launch_bounds__(TK_ENUM_NT) void tk_enum_count(GpuRoaringView v, uint64_t n_base, uint32_t* counts,
                                                            TkArgs a)
{
    tk_init_from(a, static_cast<uint64_t>(blockIdx.x) * TK_ENUM_NT + threadIdx.x,
                 static_cast<uint64_t>(gridDim.x) * TK_ENUM_NT);
    __shared__ alignas(16) uint32_t img[2048];
    __shared__ int32_t cover[2048];
    __shared__ int32_t s_c;
    __shared__ uint32_t red[TK_ENUM_NT / 64];
    const uint32_t c = block_sum<TK_ENUM_NT>(__popc(tk_enum_word(v, n_base, img, cover, &s_c)), red);
    if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

__global__ __launch_bounds__(TK_ENUM_NT) void tk_enum_write(GpuRoaringView v, uint64_t n_base, const uint32_t* counts,
                                                            uint32_t* sel, uint32_t* n_sel)
{
    __shared__ alignas(16) uint32_t img[2048];
    __shared__ int32_t cover[2048];
    __shared__ int32_t s_c;
    __shared__ uint32_t red[TK_ENUM_NT / 64];
    uint32_t pre = 0;
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += TK_ENUM_NT) pre += counts[i];
    const uint32_t run = block_sum<TK_ENUM_NT>(pre, red);
    const uint32_t word = tk_enum_word(v, n_base, img, cover, &s_c);
    uint32_t tot;
    uint32_t pos = run + block_excl_scan<TK_ENUM_NT>(__popc(word), red, tot);
    const uint32_t id0 = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * TK_ENUM_IDS) + 32u * threadIdx.x;
    for (uint32_t x = word; x; x &= x - 1) sel[pos++] = id0 + static_cast<uint32_t>(__builtin_ctz(x));
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *n_sel = run + tot;
}

// ---- 2. distances and per-chunk selection ----------------------------------

// Per-wave selection state in LDS.
struct TkWave {
    float cd[TK_CB];  // candidate buffer: distance, id, query slot (0..31)
    uint32_t cid[TK_CB];
    uint64_t sk[TK_CB];  // sort keys during a merge: query << 32 | distance bits
    float td[TK_QW];     // the query's k-th best so far (+inf, NOID while the list is short)
    float tm[TK_QW];     // the query's m_rank-th best so far (+inf while the list is shorter)
    uint32_t tid[TK_QW];
    uint32_t ln[TK_QW];   // list length
    uint32_t par[TK_QW];  // plane holding the list
    uint32_t qcnt[TK_QW];
    uint32_t qoff[TK_QW];
    uint8_t cq[TK_CB];
};

template <int DP>
struct TkLds {
    float tile[2][TK_ROWS * (DP + 4)];  // rows skewed by 16 B: conflict-free b128 reads
    float xg[2][TK_ROWS];               // (1 - TK_GATE_ERR) |x|^2, NaN for rows past the chunk
    uint32_t id[2][TK_ROWS];
    TkWave w[TK_WAVES];
    uint32_t flush_req;  // tile index at which some wave asked every wave to merge
};

__device__ __forceinline__ float tk_atomic_load(const uint32_t* p)
{
    return __uint_as_float(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Bound on the query's k-th distance from the chunks' m_rank-th distances: the
// chunks that have published one hold at least m_rank rows each at or below
// the largest of them, so once they number k / m_rank or more, that largest
// value bounds the k-th distance of the union.  The lane pair of the query
// (j, j + 32) splits the chunks between its two lanes.
__device__ __forceinline__ float tk_spread_bound(const uint32_t* tau_m, uint32_t n_chunks, uint32_t n_q, uint32_t q,
                                                 bool qok, uint32_t h, uint32_t k, uint32_t m_rank)
{
    float mx = 0.f;
    uint32_t c_fin = 0;
    if (qok) {
        for (uint32_t c = h; c < n_chunks; c += 2) {
            const float v = tk_atomic_load(tau_m + static_cast<size_t>(c) * n_q + q);
            if (v != __builtin_inff()) {
                ++c_fin;
                mx = fmaxf(mx, v);
            }
        }
    }
    c_fin += __shfl_xor(c_fin, 32, 64);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    return c_fin * m_rank >= k ? mx : __builtin_inff();
}

// Merges the wave's candidate buffer into the sorted top-k lists of its
// queries (global memory, [chunk][query][k] in two planes) and publishes every
// full list's k-th distance to the shared per-query bound.  Wave-level: no
// block barrier.  The whole buffer is sorted by (query, distance, id) in one
// bitonic network, which leaves each query's candidates as a sorted run; then
// the lane of each query walks its list (read from its current plane) and
// its run together and writes the first min(k, n + nc) of the union to the
// other plane.  Distances are non-negative, so their bits order as values.
__device__ __forceinline__ void tk_flush(TkWave& W, uint32_t cnt, uint32_t k, uint32_t m_rank, uint32_t nq_wave,
                                         float* gd_row, uint32_t* gi_row, size_t plane, uint32_t* tau_q0,
                                         uint32_t* tau_m_q0)
{
    const uint32_t lane = __lane_id();
    if (lane < TK_QW) W.qcnt[lane] = 0;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t e = lane; e < cnt; e += 64) atomicAdd(&W.qcnt[W.cq[e]], 1u);
    uint32_t P = 64;
    while (P < cnt) P <<= 1;
    for (uint32_t e = lane; e < P; e += 64) {
        if (e < cnt) {
            W.sk[e] = (static_cast<uint64_t>(W.cq[e]) << 32) | __float_as_uint(W.cd[e]);
        } else {
            W.sk[e] = ~0ull;
            W.cid[e] = TK_NOID;
        }
    }
    __builtin_amdgcn_wave_barrier();
    const uint32_t c_l = lane < TK_QW ? W.qcnt[lane] : 0u;
    const uint32_t o_l = wave_incl_scan(c_l) - c_l;
    for (uint32_t size = 2; size <= P; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t pp = lane; pp < P / 2; pp += 64) {
                const uint32_t i = 2 * stride * (pp / stride) + (pp % stride);
                const uint32_t i2 = i + stride;
                const uint64_t a0 = W.sk[i], a1 = W.sk[i2];
                const uint32_t b0 = W.cid[i], b1 = W.cid[i2];
                const bool up = (i & size) == 0;
                const bool lt = a1 < a0 || (a1 == a0 && b1 < b0);
                if (lt == up) {
                    W.sk[i] = a1;
                    W.cid[i] = b1;
                    W.sk[i2] = a0;
                    W.cid[i2] = b0;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (lane < nq_wave && c_l > 0) {
        const uint32_t n = W.ln[lane], par = W.par[lane];
        const float* ind = gd_row + par * plane + static_cast<size_t>(lane) * k;
        const uint32_t* ini = gi_row + par * plane + static_cast<size_t>(lane) * k;
        float* outd = gd_row + (par ^ 1u) * plane + static_cast<size_t>(lane) * k;
        uint32_t* outi = gi_row + (par ^ 1u) * plane + static_cast<size_t>(lane) * k;
        const uint32_t m = min(k, n + c_l);
        uint32_t ia = 0, ib = o_l;
        const uint32_t eb = o_l + c_l;
        float xa = n ? ind[0] : __builtin_inff();
        uint32_t xia = n ? ini[0] : TK_NOID;
        float yb = __uint_as_float(static_cast<uint32_t>(W.sk[ib]));
        uint32_t yib = W.cid[ib];
        float td = W.td[lane], tm = W.tm[lane];
        uint32_t tid = W.tid[lane];
        for (uint32_t r = 0; r < m; ++r) {
            const bool take_a = ia < n && (ib >= eb || tk_less(xa, xia, yb, yib));
            float d;
            uint32_t id;
            if (take_a) {
                d = xa;
                id = xia;
                if (++ia < n) {
                    xa = ind[ia];
                    xia = ini[ia];
                }
            } else {
                d = yb;
                id = yib;
                if (++ib < eb) {
                    yb = __uint_as_float(static_cast<uint32_t>(W.sk[ib]));
                    yib = W.cid[ib];
                }
            }
            outd[r] = d;
            outi[r] = id;
            if (r == k - 1) {
                td = d;
                tid = id;
            }
            if (r == m_rank - 1) tm = d;
        }
        W.td[lane] = td;
        W.tid[lane] = tid;
        W.tm[lane] = tm;
        W.ln[lane] = m;
        W.par[lane] = par ^ 1u;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < nq_wave) {
        if (W.ln[lane] == k) atomicMin(tau_q0 + lane, __float_as_uint(W.td[lane]));
        if (W.ln[lane] >= m_rank)
            __hip_atomic_store(tau_m_q0 + lane, __float_as_uint(W.tm[lane]), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    // The lists are re-read by this wave at its next merge.
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

template <int DP>
__device__ __forceinline__ void tk_load_rows(const TkArgs& a, uint64_t row0, uint64_t row_end, float4 (&pre)[DP / 32],
                                             uint32_t (&pid)[DP / 32])
{
    constexpr int TPR = DP / 4;            // threads per row (one float4 each)
    constexpr int RPP = TK_NT / TPR;       // rows per pass
    const uint32_t t = threadIdx.x;
    const uint32_t c = (t % TPR) * 4;      // first column of this thread
#pragma unroll
    for (int p = 0; p < DP / 32; ++p) {
        const uint64_t r = row0 + static_cast<uint64_t>(p * RPP + t / TPR);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        uint32_t id = TK_NOID;
        if (r < row_end) {
            id = a.sel ? a.sel[r] : static_cast<uint32_t>(r);
            const float* src = a.base + static_cast<size_t>(id) * a.dim;
            if (a.vec) {
                if (c < a.dim) v = *reinterpret_cast<const float4*>(src + c);
            } else {
                if (c + 0 < a.dim) v.x = src[c + 0];
                if (c + 1 < a.dim) v.y = src[c + 1];
                if (c + 2 < a.dim) v.z = src[c + 2];
                if (c + 3 < a.dim) v.w = src[c + 3];
            }
        }
        pre[p] = v;
        pid[p] = id;
    }
}

// The prefetch of a persistent loop, without branches or selects on loaded
// values (either makes the compiler wait for the loads where they are issued):
// the raw ids of a tile's rows, sel[min(r, last)] (or r without a filter),
// loaded a tile ahead of their use; tk_ids_valid then marks the rows past the
// tile as TK_NOID, and tk_load_rows_nb loads a row for every id (row 0 stands
// in for TK_NOID; tk_store_rows stores zeros for it).
template <int DP, bool SEL>
__device__ __forceinline__ void tk_ids_raw(const TkArgs& a, uint64_t row0, uint64_t last, uint32_t (&raw)[DP / 32])
{
    constexpr int TPR = DP / 4;
    constexpr int RPP = TK_NT / TPR;
#pragma unroll
    for (int p = 0; p < DP / 32; ++p) {
        const uint64_t r = row0 + static_cast<uint64_t>(p * RPP + threadIdx.x / TPR);
        raw[p] = SEL ? a.sel[std::min<uint64_t>(r, last)] : static_cast<uint32_t>(r);
    }
}

template <int DP>
__device__ __forceinline__ void tk_ids_valid(uint64_t row0, uint64_t row_end, uint32_t (&pid)[DP / 32])
{
    constexpr int TPR = DP / 4;
    constexpr int RPP = TK_NT / TPR;
#pragma unroll
    for (int p = 0; p < DP / 32; ++p) {
        const uint64_t r = row0 + static_cast<uint64_t>(p * RPP + threadIdx.x / TPR);
        if (r >= row_end) pid[p] = TK_NOID;
    }
}

template <int DP>
__device__ __forceinline__ void tk_load_rows_nb(const TkArgs& a, const uint32_t (&pid)[DP / 32], float4 (&pre)[DP / 32])
{
    constexpr int TPR = DP / 4;
    const uint32_t c = (threadIdx.x % TPR) * 4;
#pragma unroll
    for (int p = 0; p < DP / 32; ++p) {
        const uint32_t id = pid[p] != TK_NOID ? pid[p] : 0u;
        const float* src = a.base + static_cast<size_t>(id) * a.dim;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (a.vec) {
            if (c < a.dim) v = *reinterpret_cast<const float4*>(src + c);
        } else {
            if (c + 0 < a.dim) v.x = src[c + 0];
            if (c + 1 < a.dim) v.y = src[c + 1];
            if (c + 2 < a.dim) v.z = src[c + 2];
            if (c + 3 < a.dim) v.w = src[c + 3];
        }
        pre[p] = v;
    }
}

// Sum over aligned groups of W lanes (8, 16 or 32) with DPP moves, no LDS
// round trips: quad swaps, the half-row and row mirrors, then (W = 32) row
// 15's value broadcast into the next row.  Every lane of a group holds the
// total for W <= 16, the group's upper 16 lanes for W = 32.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float tk_dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, false));
}

template <int W>
__device__ __forceinline__ float tk_group_sum(float x)
{
    static_assert(W == 8 || W == 16 || W == 32, "lane groups of 8, 16 or 32");
    x += tk_dpp<0xB1, 0xF>(x);   // quad_perm [1, 0, 3, 2]
    x += tk_dpp<0x4E, 0xF>(x);   // quad_perm [2, 3, 0, 1]
    x += tk_dpp<0x141, 0xF>(x);  // row_half_mirror
    if constexpr (W >= 16) x += tk_dpp<0x140, 0xF>(x);  // row_mirror
    if constexpr (W == 32) x += tk_dpp<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3 (rows 0 and 2 add 0)
    return x;
}

template <int DP, class Lds>
__device__ __forceinline__ void tk_store_rows(Lds& L, int buf, const float4 (&pre)[DP / 32],
                                              const uint32_t (&pid)[DP / 32])
{
    constexpr int TPR = DP / 4;
    constexpr int RPP = TK_NT / TPR;
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int p = 0; p < DP / 32; ++p) {
        const int row = p * RPP + static_cast<int>(t / TPR);
        const int c = static_cast<int>(t % TPR) * 4;
        const float4 v = pid[p] != TK_NOID ? pre[p] : make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(&L.tile[buf][row * (DP + 4) + c]) = v;
        const float ss = tk_group_sum<TPR>(v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w);
        if (static_cast<int>(t % TPR) == (TPR == 32 ? TPR - 1 : 0)) {  // a lane holding the row's total
            L.xg[buf][row] = pid[p] != TK_NOID ? (1.f - TK_GATE_ERR) * ss : __builtin_nanf("");
            L.id[buf][row] = pid[p];
        }
    }
}

// This lane's query dimensions [h DP/2, h DP/2 + DP/2) into qreg (zeros past
// dim or for a lane without a query): 16-byte loads when the queries allow
// them, each a contiguous 16 bytes of the lane's row, else one float at a
// time.  Returns the sum of their squares.
template <int DP>
__device__ __forceinline__ float tk_load_query(const TkArgs& a, bool qok, uint32_t q, uint32_t h, float (&qreg)[DP / 2])
{
    const float* src = a.queries + static_cast<size_t>(q) * a.dim + h * (DP / 2);
    if (a.qvec) {
#pragma unroll
        for (int s = 0; s < DP / 2; s += 4) {
            const uint32_t c = h * (DP / 2) + s;
            const float4 v = (qok && c < a.dim) ? *reinterpret_cast<const float4*>(src + s) : make_float4(0.f, 0.f, 0.f, 0.f);
            qreg[s] = v.x, qreg[s + 1] = v.y, qreg[s + 2] = v.z, qreg[s + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int s = 0; s < DP / 2; ++s) {
            const uint32_t c = h * (DP / 2) + s;
            qreg[s] = (qok && c < a.dim) ? src[s] : 0.f;
        }
    }
    float part = 0.f;
#pragma unroll
    for (int s = 0; s < DP / 2; ++s) part += qreg[s] * qreg[s];
    return part;
}

// Base row held by accumulator register rr (0..31: block rr/16, register
// rr%16) of the lane half hh.
__device__ __forceinline__ int tk_row(int rr, int hh)
{
    return (rr >> 4) * 32 + 8 * ((rr & 15) >> 2) + 4 * hh + (rr & 3);
}

template <int DP, bool SEL>
__global__ __launch_bounds__(TK_NT) void tk_dist(TkArgs a)
{
    __shared__ TkLds<DP> L;
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t h = lane >> 5;    // lane half: which half of the dimensions it feeds
    const uint32_t j = lane & 31u;   // query column of this lane
    TkWave& W = L.w[wave];

    // Blocks are dispatched round-robin over the 8 XCDs: the blocks of one XCD
    // take consecutive query blocks of the same chunks, so they share the
    // chunk's base rows in that XCD's L2.
    const uint32_t n_qb = (a.n_q + TK_QB - 1) / TK_QB;
    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t pidx = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    const uint32_t chunk = pidx / n_qb;
    const uint32_t qb = pidx % n_qb;

    const uint64_t n_rows = tk_rows(a);
    if (a.gate && (n_rows <= a.keep || !a.qb_over[qb])) return;  // tk_select has answered
    const uint64_t rpc = ((n_rows + a.n_chunks - 1) / a.n_chunks + TK_ROWS - 1) / TK_ROWS * TK_ROWS;
    const uint64_t r0 = std::min<uint64_t>(n_rows, static_cast<uint64_t>(chunk) * rpc);
    const uint64_t r1 = std::min<uint64_t>(n_rows, r0 + rpc);
    const uint32_t n_tiles = static_cast<uint32_t>((r1 - r0 + TK_ROWS - 1) / TK_ROWS);

    const uint32_t q0 = qb * TK_QB + wave * TK_QW;
    const uint32_t nq_wave = q0 < a.n_q ? std::min<uint32_t>(TK_QW, a.n_q - q0) : 0u;
    // After candidates the list path answers the queries whose lists overflowed;
    // the block's others have no state here and take no part.
    const bool qok = j < nq_wave && (!a.gate || a.q_over[q0 + j]);
    const bool busy = __ballot(qok) != 0;  // wave-uniform
    const size_t list_row = (static_cast<size_t>(chunk) * a.n_q + q0) * a.k;
    uint32_t* tau_q0 = a.tau + q0;
    uint32_t* tau_m_q0 = a.tau_m + static_cast<size_t>(chunk) * a.n_q + q0;

    if (lane < TK_QW) {
        W.td[lane] = __builtin_inff();
        W.tm[lane] = __builtin_inff();
        W.tid[lane] = TK_NOID;
        W.ln[lane] = 0;
        W.par[lane] = 0;
    }
    if (threadIdx.x == 0) L.flush_req = TK_NOID;

    // B operand: this lane's query, dimensions [h*DP/2, h*DP/2 + DP/2).
    float qreg[DP / 2];
    const float qpart = tk_load_query<DP>(a, qok, q0 + j, h, qreg);
    const float qg = (1.f - TK_GATE_ERR) * (qpart + __shfl_xor(qpart, 32, 64));

    // The prefetch as in tk_est: tile t + 1's rows (ids known since tile
    // t - 1) and tile t + 2's raw ids are issued before tile t's MFMA and
    // waited for after it.
    auto tile_r0 = [&](uint32_t i) { return r0 + static_cast<uint64_t>(i) * TK_ROWS; };
    auto tile_r1 = [&](uint32_t i) { return std::min<uint64_t>(r1, tile_r0(i) + TK_ROWS); };
    const uint64_t last = n_rows > 0 ? n_rows - 1 : 0;
    float4 pre[DP / 32];
    uint32_t pid[DP / 32], nid[DP / 32];
    if constexpr (SEL) {
        if (n_rows > 0) tk_ids_raw<DP, SEL>(a, tile_r0(1), last, nid);
    }
    if (n_tiles > 0) {
        tk_load_rows<DP>(a, r0, r1, pre, pid);
        tk_store_rows<DP>(L, 0, pre, pid);
    }
    if constexpr (SEL) {
#pragma unroll
        for (int p = 0; p < DP / 32; ++p) pid[p] = n_rows > 0 ? nid[p] : TK_NOID;
        tk_ids_valid<DP>(tile_r0(1), tile_r1(1), pid);
    }
    __syncthreads();

    // Thresholds of this lane's query: the own list's k-th best (td, tidv) and
    // the bound shared by all chunks (tsh).  A row whose distance exceeds
    // either cannot be in the answer.
    float td = __builtin_inff();
    uint32_t tidv = TK_NOID;
    float tsh = __builtin_inff();
    float seed = __builtin_inff();  // bound on the chunk's k-th best from its first tile
    uint32_t cnt = 0;  // wave-uniform fill of the candidate buffer
    for (uint32_t t = 0; t < n_tiles; ++t) {
        const int b = static_cast<int>(t & 1u);
        if constexpr (SEL) {
            tk_load_rows_nb<DP>(a, pid, pre);
            tk_ids_raw<DP, SEL>(a, tile_r0(t + 2), last, nid);
        } else if (t + 1 < n_tiles) {  // the row numbers are the ids
            tk_load_rows<DP>(a, tile_r0(t + 1), r1, pre, pid);
        }
        const float tsh_new = qok ? tk_atomic_load(tau_q0 + j) : __builtin_inff();

        if (busy) {
            f32x16 acc0 = {}, acc1 = {};
            const float* A0 = &L.tile[b][j * (DP + 4) + h * (DP / 2)];
            const float* A1 = A0 + 32 * (DP + 4);
#pragma unroll
            for (int s = 0; s < DP / 2; s += 4) {
                const float4 x0 = *reinterpret_cast<const float4*>(A0 + s);
                const float4 x1 = *reinterpret_cast<const float4*>(A1 + s);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x0.x, qreg[s + 0], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(x1.x, qreg[s + 0], acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x0.y, qreg[s + 1], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(x1.y, qreg[s + 1], acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x0.z, qreg[s + 2], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(x1.z, qreg[s + 2], acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x0.w, qreg[s + 3], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(x1.w, qreg[s + 3], acc1, 0, 0, 0);
            }
            tsh = fminf(tsh, tsh_new);
            // Gate: the MFMA distance |q|^2 + |x|^2 - 2 q.x lies within
            // TK_GATE_ERR (|q|^2 + |x|^2) of the fp32 direct distance, so a
            // row passes when that margin could put it at or below the
            // thresholds.  Accumulator register r of block u holds base row
            // tk_row(16u + r, h) against query column j.
            // The accumulators become the estimates |q|^2 + |x|^2 - 2 q.x
            // (scaled as above; NaN for rows past the chunk).
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                const float4 g0 = *reinterpret_cast<const float4*>(&L.xg[b][8 * rq + 4 * h]);
                const float4 g1 = *reinterpret_cast<const float4*>(&L.xg[b][32 + 8 * rq + 4 * h]);
                acc0[4 * rq + 0] = qg + g0.x - 2.f * acc0[4 * rq + 0];
                acc0[4 * rq + 1] = qg + g0.y - 2.f * acc0[4 * rq + 1];
                acc0[4 * rq + 2] = qg + g0.z - 2.f * acc0[4 * rq + 2];
                acc0[4 * rq + 3] = qg + g0.w - 2.f * acc0[4 * rq + 3];
                acc1[4 * rq + 0] = qg + g1.x - 2.f * acc1[4 * rq + 0];
                acc1[4 * rq + 1] = qg + g1.y - 2.f * acc1[4 * rq + 1];
                acc1[4 * rq + 2] = qg + g1.z - 2.f * acc1[4 * rq + 2];
                acc1[4 * rq + 3] = qg + g1.w - 2.f * acc1[4 * rq + 3];
            }
            if (t == 0 && a.k <= TK_ROWS) {
                // Seed: the k-th smallest estimate of the first tile's rows
                // (bisection on the lane pair's 64 estimates), raised to an
                // upper estimate, bounds the chunk's k-th best distance, so
                // the first tile yields about k candidates per query instead
                // of all of its rows.
                float lo = __builtin_inff(), hi = -__builtin_inff();
                uint32_t nv = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float e0 = acc0[r], e1 = acc1[r];
                    if (e0 == e0) {
                        lo = fminf(lo, e0);
                        hi = fmaxf(hi, e0);
                        ++nv;
                    }
                    if (e1 == e1) {
                        lo = fminf(lo, e1);
                        hi = fmaxf(hi, e1);
                        ++nv;
                    }
                }
                lo = fminf(lo, __shfl_xor(lo, 32, 64));
                hi = fmaxf(hi, __shfl_xor(hi, 32, 64));
                nv += __shfl_xor(nv, 32, 64);
                float xgmax = L.xg[b][lane];
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) xgmax = fmaxf(xgmax, __shfl_xor(xgmax, o, 64));
                const bool do_seed = qok && nv >= a.k;
                for (int it = 0; it < 24; ++it) {  // invariant: at least k estimates <= hi
                    const float mid = 0.5f * (lo + hi);
                    uint32_t c = 0;
#pragma unroll
                    for (int r = 0; r < 16; ++r) c += (acc0[r] <= mid ? 1u : 0u) + (acc1[r] <= mid ? 1u : 0u);
                    c += __shfl_xor(c, 32, 64);
                    if (c >= a.k)
                        hi = mid;
                    else
                        lo = mid;
                }
                if (do_seed) seed = hi + TK_SEED_ERR * (qg + xgmax);
            }
            const float tgate = fminf(fminf(td, tsh), seed);
            uint32_t pm = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                pm |= (acc0[r] <= tgate ? 1u : 0u) << r;
                pm |= (acc1[r] <= tgate ? 1u : 0u) << (16 + r);
            }
            if (!qok) pm = 0;
            if (__ballot(pm != 0)) {
                // Both lanes of a query (j and j + 32) walk the query's gated
                // rows in the same order; each sums its half of the dimensions
                // and the pair adds the halves.
                uint32_t m0 = __shfl(pm, static_cast<int>(j), 64);
                uint32_t m1 = __shfl(pm, static_cast<int>(j + 32), 64);
                while (__ballot((m0 | m1) != 0)) {
                    if (cnt + TK_QW > TK_CB) {
                        tk_flush(W, cnt, a.k, a.m_rank, nq_wave, a.list_d + list_row, a.list_id + list_row, a.plane, tau_q0, tau_m_q0);
                        cnt = 0;
                        td = W.td[j];
                        tidv = W.tid[j];
                        if (qok) tsh = fminf(tsh, tk_atomic_load(tau_q0 + j));
                        tsh = fminf(tsh, tk_spread_bound(a.tau_m, a.n_chunks, a.n_q, q0 + j, qok, h, a.k, a.m_rank));
                    }
                    int row = -1;
                    if (m0) {
                        row = tk_row(__builtin_ctz(m0), 0);
                        m0 &= m0 - 1;
                    } else if (m1) {
                        row = tk_row(__builtin_ctz(m1), 1);
                        m1 &= m1 - 1;
                    }
                    float e2 = 0.f;
                    if (row >= 0) {
                        const float* xr = &L.tile[b][row * (DP + 4) + h * (DP / 2)];
#pragma unroll
                        for (int s2 = 0; s2 < DP / 2; s2 += 4) {
                            const float4 v = *reinterpret_cast<const float4*>(xr + s2);
                            float e;
                            e = qreg[s2 + 0] - v.x; e2 = fmaf(e, e, e2);
                            e = qreg[s2 + 1] - v.y; e2 = fmaf(e, e, e2);
                            e = qreg[s2 + 2] - v.z; e2 = fmaf(e, e, e2);
                            e = qreg[s2 + 3] - v.w; e2 = fmaf(e, e, e2);
                        }
                    }
                    const float d = e2 + __shfl_xor(e2, 32, 64);
                    bool f = false;
                    uint32_t id = 0;
                    if (h == 0 && row >= 0) {
                        id = L.id[b][row];
                        f = tk_less(d, id, td, tidv) && d <= tsh && d <= seed;
                    }
                    const uint64_t m = __ballot(f);
                    if (f) {
                        const uint32_t pos = cnt + static_cast<uint32_t>(__popcll(m & lanemask_lt()));
                        W.cd[pos] = d;
                        W.cid[pos] = id;
                        W.cq[pos] = static_cast<uint8_t>(j);
                    }
                    cnt += static_cast<uint32_t>(__popcll(m));
                }
            }
        }
        // Merges are taken together: a wave whose buffer is half full asks
        // every wave to merge after the barrier, so the waves of the block
        // stall for one merge at a time rather than one after another.
        if (cnt > TK_CB * 3 / 4 && lane == 0) L.flush_req = t;
        if constexpr (SEL) {
            tk_store_rows<DP>(L, b ^ 1, pre, pid);
#pragma unroll
            for (int p = 0; p < DP / 32; ++p) pid[p] = nid[p];
            tk_ids_valid<DP>(tile_r0(t + 2), tile_r1(t + 2), pid);
        } else if (t + 1 < n_tiles) {
            tk_store_rows<DP>(L, b ^ 1, pre, pid);
        }
        __syncthreads();
        if (L.flush_req == t && cnt > 0) {
            tk_flush(W, cnt, a.k, a.m_rank, nq_wave, a.list_d + list_row, a.list_id + list_row, a.plane, tau_q0, tau_m_q0);
            cnt = 0;
            td = W.td[j];
            tidv = W.tid[j];
            if (qok) tsh = fminf(tsh, tk_atomic_load(tau_q0 + j));
        }
        if (busy && (t & 7u) == 7u)
            tsh = fminf(tsh, tk_spread_bound(a.tau_m, a.n_chunks, a.n_q, q0 + j, qok, h, a.k, a.m_rank));
    }
    if (nq_wave > 0) {
        if (cnt) tk_flush(W, cnt, a.k, a.m_rank, nq_wave, a.list_d + list_row, a.list_id + list_row, a.plane, tau_q0, tau_m_q0);
        __builtin_amdgcn_wave_barrier();
        if (lane < nq_wave) a.list_n[static_cast<size_t>(chunk) * a.n_q + q0 + lane] = W.ln[lane] | (W.par[lane] << 31);
    }
}

// ---- 3. merge of the chunk lists -------------------------------------------

__global__ __launch_bounds__(TK_MERGE_NT) void tk_merge(TkArgs a, const float* list_d, const uint32_t* list_id,
                                                         size_t plane, const uint32_t* list_n, uint32_t n_chunks,
                                                         uint32_t n_q, uint32_t k, float* out_d, int64_t* out_id)
{
    if (tk_small(a, tk_rows(a))) return;  // tk_select has answered
    constexpr int W = TK_MERGE_NT / 64;
    __shared__ float ad[W][2][TK_KMAX];
    __shared__ uint32_t ai[W][2][TK_KMAX];
    __shared__ float cd[W][TK_KMAX];
    __shared__ uint32_t ci[W][TK_KMAX];
    const uint32_t lane = __lane_id();
    const uint32_t w = threadIdx.x >> 6;
    const uint32_t q = blockIdx.x * W + w;
    if (q >= n_q) return;  // whole wave; no block barrier below
    if (a.gate && !a.q_over[q]) return;
    uint32_t n = 0;
    int cur = 0;
    // The next chunk's list is loaded into registers (k <= 256: four entries a
    // lane) while the current one is merged.
    constexpr int PER = TK_KMAX / 64;
    float nd[PER];
    uint32_t ni[PER], nm = 0;
    auto fetch = [&](uint32_t c) {
        const size_t row = static_cast<size_t>(c) * n_q + q;
        const uint32_t ln = list_n[row];
        nm = ln & 0x7FFFFFFFu;
        const size_t base = (ln >> 31) * plane + row * k;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const uint32_t i = lane + 64u * e;
            nd[e] = i < nm ? list_d[base + i] : 0.f;
            ni[e] = i < nm ? list_id[base + i] : 0u;
        }
    };
    if (n_chunks) fetch(0);
    for (uint32_t c = 0; c < n_chunks; ++c) {
        const uint32_t m = nm;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const uint32_t i = lane + 64u * e;
            if (i < m) {
                cd[w][i] = nd[e];
                ci[w][i] = ni[e];
            }
        }
        if (c + 1 < n_chunks) fetch(c + 1);
        if (m == 0) continue;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t i = lane; i < n; i += 64) {
            const float x = ad[w][cur][i];
            const uint32_t xi = ai[w][cur][i];
            const uint32_t r = i + tk_lower_bound(cd[w], ci[w], m, x, xi);
            if (r < k) {
                ad[w][cur ^ 1][r] = x;
                ai[w][cur ^ 1][r] = xi;
            }
        }
        for (uint32_t e = lane; e < m; e += 64) {
            const float y = cd[w][e];
            const uint32_t yi = ci[w][e];
            const uint32_t r = e + tk_lower_bound(ad[w][cur], ai[w][cur], n, y, yi);
            if (r < k) {
                ad[w][cur ^ 1][r] = y;
                ai[w][cur ^ 1][r] = yi;
            }
        }
        __builtin_amdgcn_wave_barrier();
        n = min(k, n + m);
        cur ^= 1;
    }
    for (uint32_t r = lane; r < k; r += 64) {
        out_d[static_cast<size_t>(q) * k + r] = r < n ? ad[w][cur][r] : __builtin_inff();
        out_id[static_cast<size_t>(q) * k + r] = r < n ? static_cast<int64_t>(ai[w][cur][r]) : int64_t(-1);
    }
}

// ---- 2b. estimates on split f16 MFMA --------------------------------------------
// q.x from f16 halves: a row is scaled by a power of two that brings its norm
// into [2^14, 2^15), then x = hi + lo with hi = f16(x) and lo = f16(x - hi), and
// the same for the query; hi.hi + lo.hi + hi.lo accumulate in fp32 in one MFMA
// chain.  The remainders are 2^-22 of an element (2^-29 of the row's norm where
// lo is below f16's normal range), under the fp32 accumulation's own rounding;
// v_mfma_f32_32x32x16_f16 runs at 16 times the fp32 MFMA rate, so three of them
// cost 3/16 of the fp32 product.
//
// A rank-2 product (one fp32 MFMA) then brings the accumulator to
//   sx sq (2 q.x - |x|^2 - |q|^2 + gate) / 2
// (sx, sq the scales; the norms shrunk by 1 - TK_EST_ERR): a row can lie at or
// below the query's gate exactly when it is >= 0, one maximum over the
// accumulator's registers and one test per 32 x 32 pairs.  With gate = 0 it is
// the estimate times -sx sq / 2.  The norms come last so that the products are
// rounded at their own size, as an fp32 MFMA's are before its norms are added.
//
// For candidates the accumulator first holds hi.hi alone, whose distance from
// q.x is bounded (TK_COARSE_ERR): the rank-2 test with that much added excludes
// most 32 x 32 fragments, and only the others compute the cross products.
//
// A workgroup's waves are QG query groups of 32 QW queries (their hi halves live
// in registers) by two row groups of 32 rows; a tile of 64 rows goes through
// LDS once for all of them.  The next tile's split (its norms, scales and
// halves, ~150 vector instructions a lane) is cut into pieces that run between
// the current tile's MFMAs, and rows are loaded two tiles ahead.  Large query
// counts take 256 queries a workgroup (QW 2, QG 4, eight waves, one a CU): the
// tile's split and its reads are then shared by 256.  Up to 64 queries are bound
// by reading the rows (QW 1, QG 2, four waves): two workgroups a CU, which do
// not wait for each other's loads; so are sets whose estimates are all kept.
// Of the variants, QW 1's candidates of 97 to 128 dimensions with scalar row loads
// spill (5 to 13 registers, compiler's report).
// Measured (128 dimensions, 1024 queries, k 10, both stages of candidates): 550 us
// for 822K of 10M rows, 1814 us for 4M unfiltered ones, against 2505 us and ~9.5 ms
// of fp32 MFMA with sorted lists.  All three products for every pair took 706 us
// of 1M rows when the test on hi.hi came in at 483 (the MFMAs alone 480: 1.6
// PFLOP/s, where the clock gives way to power).  64 queries: 4M rows 372 us (5.5
// TB/s of rows), 300K x 100 36 us.
// The estimate's error against fp64, 32 x 32 blocks of 17 to 128 dimensions
// (normal, positive, and over 2^20 of magnitudes), rms of |q|^2 + |x|^2:
// 5.5e-8 to 1.45e-7, with fp32 MFMA 6.4e-8 to 1.73e-7 (lower in each block).
constexpr uint32_t TK_KEEP = 16384;         // rows whose estimates are all kept, and the sample, at most ...
constexpr uint32_t TK_KEEP_MAX[] = {24576, 40960, 65536};  // ... rows kept where that is all of a call's rows
constexpr uint32_t TK_SCRATCH = 1u << 30;   // bytes of estimates, and of candidate lists, at most
// Candidates a query's lists hold together: every row up to TK_CAND_WHOLE, else TK_CAND_MANY (or eight times those
// expected) and at most TK_CAND_CAP a list.
constexpr uint32_t TK_CAND_WHOLE = 1u << 21;
constexpr uint32_t TK_CAND_MANY = 1u << 18;
constexpr uint32_t TK_CAND_CAP = 2048;
constexpr double TK_TWO_STAGE = 1024;       // expected candidates of a query, and of all of them, above which a
constexpr double TK_TWO_STAGE_ALL = 1 << 17;  // second bound pays
// |q.x - hi.hi| <= (2 x 2^-11 + 2^-22) |q||x|, and 2 |q||x| <= |q|^2 + |x|^2: the
// test on hi.hi with the norms shrunk by TK_COARSE_ERR more excludes only pairs
// that the full estimate excludes (2% covers its rounding).
constexpr float TK_COARSE_ERR = 1.02f * 0x1p-10f;
constexpr float TK_COARSE = 1.f - TK_COARSE_ERR;
constexpr float TK_GATE_ROUND = 0x1p-20f;   // rounding of a stored estimate, relative to the gate

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));  // (a float4 struct's load is split where two paths merge)

template <int KS, int QW, int QG>
struct TkEst {
    static constexpr int RG = 2;
    static constexpr int WAVES = RG * QG;
    static constexpr int NT = 64 * WAVES;
    static constexpr int T = 32 * RG;         // rows of a tile
    static constexpr int QB = 32 * QW * QG;   // queries of a workgroup
    static constexpr int DP = 16 * KS;        // padded dimensions
    // Eight threads load a row, a float4 of each 32 dimensions (whole 128-byte
    // lines); more threads a row would spend more on its norm and scale than
    // on its elements.
    static constexpr int TPR = 8;
    static constexpr int V = DP / 8;          // elements a thread
    static constexpr int RPP = NT / TPR;      // rows per pass
    static constexpr int P = T / RPP;         // passes
    static constexpr int RS = DP + 8;         // row stride in LDS: conflict-free 16-byte reads
};

struct alignas(16) TkRow {
    float u, z;  // the rank-2 product's row factors: -sx |x|^2 / 2 and sx
    float isx;   // 1 / sx
    uint32_t id;
};

template <int KS, int QW, int QG>
struct TkEstLds {
    using C = TkEst<KS, QW, QG>;
    alignas(16) _Float16 hi[C::T * C::RS];
    alignas(16) _Float16 lo[C::T * C::RS];
    TkRow row[C::T];
};

// What the candidates need beside it.  A wave appends its candidates to a
// buffer and writes them to their lists when it is nearly full: a store to
// memory in the tile loop would make the next wait for a tile's rows wait for
// the store too (both count in order).
template <int QB, int WAVES>
struct TkGateLds {
    static constexpr uint32_t WB = 192;  // entries a wave (LDS left by the tiles)
    float2 gq[QB];  // an estimate is gq.x - acc gq.y / sx
    uint32_t cnt[QB];
    uint2 buf[WAVES][WB];     // (estimate bits, id)
    uint16_t lq[WAVES][WB];    // query within the workgroup
};

// Scale for a squared norm: the power of two that brings the norm into
// [2^14, 2^15).  Norms outside [2^-30, 2^30] (zero aside, whose scale is 1) are
// not estimated: `odd`.
__device__ __forceinline__ float tk_scale(float ss, float& inv, bool& odd)
{
    const uint32_t e = __float_as_uint(ss) >> 23;  // ss >= 0: its biased exponent (NaN: past the range)
    odd = ss != 0.f && (e < 127u - 60u || e > 127u + 60u);
    const bool unit = odd || ss == 0.f;
    const uint32_t sh = (e + 1u) >> 1;  // floor(log2 ss / 2) + 64, for the odd bias
    const uint32_t se = unit ? 127u : 127u + 14u + 64u - sh;
    inv = __uint_as_float((254u - se) << 23);
    return __uint_as_float(se << 23);
}

// v_mul_legacy_f32: 0 times anything (infinities and NaN too) is 0.
extern "C" __device__ float tk_mul_legacy(float, float) __asm("llvm.amdgcn.fmul.legacy");

// hi and lo halves of two scaled values.
__device__ __forceinline__ void tk_split(float a, float b, f16x2& hi, f16x2& lo)
{
    const f32x2 v = {a, b};
    hi = __builtin_convertvector(v, f16x2);
    // a - hi in one instruction each (v_fma_mix_f32 reads a 16-bit half in place)
    f32x2 r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r.x) : "v"(hi), "v"(a));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r.y) : "v"(hi), "v"(b));
    lo = __builtin_convertvector(r, f16x2);
}

// Which rows a launch covers: every row or the sample (row i stands for
// i * rows / sample), and which tiles of them.
struct TkSpan {
    uint64_t rows;   // the set's
    uint64_t n;      // rows of this launch
    uint32_t lg;     // log2 of the sample's size, 0 for every row
};

// Ids of a tile's rows [r0, r0 + T) of the launch's sp.n (past the last: the last's).
template <class C, bool SEL, bool SAMPLE>
__device__ __forceinline__ void tk_est_ids(const TkArgs& a, const TkSpan& sp, uint64_t r0, uint32_t (&raw)[C::P])
{
    const uint32_t at = static_cast<uint32_t>(std::min<uint64_t>(r0, sp.n - 1));
    const uint32_t left = static_cast<uint32_t>(sp.n - 1) - at;
#pragma unroll
    for (int p = 0; p < C::P; ++p) {
        uint32_t r = at + min(p * C::RPP + threadIdx.x / C::TPR, left);
        if (SAMPLE && sp.lg) r = static_cast<uint32_t>((static_cast<uint64_t>(r) * sp.rows) >> sp.lg);
        raw[p] = SEL ? a.sel[r] : r;
    }
}

// Dimension of element e of a thread's row.
template <class C>
__device__ __forceinline__ uint32_t tk_est_col(int e)
{
    return 32u * (e / 4) + (threadIdx.x % C::TPR) * 4u + (e & 3u);
}

// Dimension at position 8 i + e of a split row in LDS, and of the queries'
// operand: the eight values that a thread stores at once are its float4s of two
// 32-dimension groups; a last odd group keeps its order.
template <int DP>
__device__ __forceinline__ uint32_t tk_est_dim(uint32_t i, uint32_t e)
{
    return i < DP / 64 * 8u ? (i / 8) * 64u + (i % 8) * 4u + 32u * (e / 4) + (e & 3u) : 8u * i + e;
}

// A thread's elements of its rows.  Dimensions past dim repeat valid ones: the
// norm leaves them out, and the queries hold zeros there.
template <class C, bool VEC>
__device__ __forceinline__ void tk_est_rows(const TkArgs& a, const uint32_t (&id)[C::P], float (&pre)[C::P][C::V])
{
#pragma unroll
    for (int p = 0; p < C::P; ++p) {
        const float* src = a.base + static_cast<size_t>(id[p]) * a.dim;
        if constexpr (VEC) {
#pragma unroll
            for (int e = 0; e < C::V; e += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(src + min(tk_est_col<C>(e), a.dim - 4u));
                pre[p][e] = v.x, pre[p][e + 1] = v.y, pre[p][e + 2] = v.z, pre[p][e + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < C::V; ++e) pre[p][e] = src[min(tk_est_col<C>(e), a.dim - 1u)];
        }
    }
}

// A tile's rows from registers into an LDS buffer, split, in PIECES steps of a
// few vector instructions that the tile loop puts between MFMAs: per pass
// V / 4 for the norm's partial sums, one for the sum over the row's threads,
// one for the scale, V / 2 that split two elements each, one for the record.
template <class C, bool VEC>
struct TkSplit {
    static constexpr int PER = C::V / 4 + 2 + C::V / 2 + 1;
    static constexpr int PIECES = C::P * PER;
    float ss, unit, inv, sx;
    bool odd;
    f16x8 hv, lv;

    template <class Buf>
    __device__ __forceinline__ void piece(int i, Buf& B, const float (&pre)[C::P][C::V], const uint32_t (&id)[C::P],
                                          uint32_t valid, uint32_t dim)
    {
        const uint32_t l = threadIdx.x % C::TPR;
        const int p = i / PER, k = i % PER;
        const uint32_t row = p * C::RPP + threadIdx.x / C::TPR;
        if (k < C::V / 4) {
            if (k == 0) ss = 0.f;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = VEC || tk_est_col<C>(4 * k + e) < dim ? pre[p][4 * k + e] : 0.f;
            const float s4 = fmaf(x[0], x[0], x[1] * x[1]) + fmaf(x[2], x[2], x[3] * x[3]);
            ss += !VEC || tk_est_col<C>(4 * k) < dim ? s4 : 0.f;
        } else if (k == C::V / 4) {
            ss = tk_group_sum<8>(ss);
        } else if (k == C::V / 4 + 1) {
            unit = tk_scale(ss, inv, odd);
            sx = odd ? 0.f : unit;  // rows that are not estimated multiply as zeros ...
        } else if (k < PER - 1) {
            const int e = 2 * (k - C::V / 4 - 2);
            f16x2 hi, lo;
            tk_split(tk_mul_legacy(pre[p][e], sx), tk_mul_legacy(pre[p][e + 1], sx), hi, lo);
            hv[e & 7] = hi.x, hv[(e & 7) + 1] = hi.y, lv[e & 7] = lo.x, lv[(e & 7) + 1] = lo.y;
            if ((e & 7) == 6) {
                const uint32_t at = row * C::RS + 8u * l + 8u * (e & ~7);
                *reinterpret_cast<f16x8*>(&B.hi[at]) = hv;
                *reinterpret_cast<f16x8*>(&B.lo[at]) = lv;
            } else if (e == C::V - 2) {  // an odd group
                const uint32_t at = row * C::RS + 4u * l + 8u * (e & ~7);
                *reinterpret_cast<f16x4*>(&B.hi[at]) = __builtin_shufflevector(hv, hv, 0, 1, 2, 3);
                *reinterpret_cast<f16x4*>(&B.lo[at]) = __builtin_shufflevector(lv, lv, 0, 1, 2, 3);
            }
        } else {
            // ... and their factor makes them pass every gate, or (past the last
            // row) none.  Thread l writes word l % 4 of the row's record.
            const float u = row >= valid ? -__builtin_inff()
                                         : odd ? __builtin_inff() : -0.5f * (1.f - TK_EST_ERR) * ss * sx;
            uint32_t w0 = __float_as_uint(u), w1 = __float_as_uint(unit), w2 = __float_as_uint(inv), w3 = id[p];
            asm("" : "+v"(w0), "+v"(w1), "+v"(w2), "+v"(w3));  // selects, not branches, which would end the block
            const uint32_t lo = (l & 1u) ? w1 : w0, hi = (l & 1u) ? w3 : w2;
            reinterpret_cast<uint32_t*>(&B.row[row])[l & 3u] = (l & 2u) ? hi : lo;
        }
    }
};

// GATE false: estimates of a small set or of the sample, into pd.  GATE true:
// candidates of a larger set; `stage` 0 takes every tile, 1 every 16th, 2 the
// others (the counts then continue).
constexpr uint32_t TK_STAGE = 16;

template <int KS, int QW, int QG, bool SEL, bool VEC, bool GATE>
__global__ __launch_bounds__((TkEst<KS, QW, QG>::NT)) __attribute__((amdgpu_waves_per_eu(2))) void tk_est(TkArgs a, uint32_t n_qb, uint32_t stage)
{
    using C = TkEst<KS, QW, QG>;
    const uint64_t rows = tk_rows(a);
    const bool small = rows <= a.keep;
    if (rows == 0 || (GATE && small)) return;
    TkSpan sp;
    sp.rows = rows;
    sp.lg = !GATE && !small && rows > a.sample ? a.sample_lg : 0u;
    sp.n = sp.lg ? a.sample : rows;
    // The workgroups of a query block take its tiles in turn.  Blocks are
    // dispatched round-robin over the 8 XCDs: an XCD's blocks take consecutive
    // query blocks of the same tiles, which then share the rows in its L2.
    const uint32_t pidx = (blockIdx.x % 8u) * (gridDim.x / 8u) + blockIdx.x / 8u;
    const uint32_t chunk = pidx / n_qb, qb = pidx % n_qb;
    if (chunk >= a.n_cw) return;
    if (GATE && !a.list_off) {
        const uint32_t q = qb * C::QB + threadIdx.x;
        if (!__syncthreads_or(threadIdx.x < C::QB && q < a.n_q && a.gate_at[q] > -__builtin_inff()))
            return;  // the list path answers the whole block
    }
    const uint64_t all = (sp.n + C::T - 1) / C::T;
    const uint64_t first = (all + TK_STAGE - 1) / TK_STAGE;  // tiles of stage 1
    const uint64_t part = stage == 0 ? all : stage == 1 ? first : all - first;
    const uint32_t n_tiles = chunk < part ? static_cast<uint32_t>((part - chunk + a.n_cw - 1) / a.n_cw) : 0u;
    const uint32_t mul = stage == 1 ? TK_STAGE : 1u;
    auto tile_r0 = [&](uint32_t i) -> uint64_t {  // first row of the workgroup's tile i
        const uint32_t g = chunk + i * a.n_cw;
        return static_cast<uint64_t>(g * mul + (stage == 2 ? g / (TK_STAGE - 1) + 1u : 0u)) * C::T;
    };
    // Two tiles, as objects of their own: writes to one may pass reads of the other.
    __shared__ TkEstLds<KS, QW, QG> T0, T1;
    __shared__ alignas(16) float s_isq[C::QB];
    // Candidates are found about the query block's centre.
    __shared__ alignas(16) float s_centre[GATE ? C::DP : 4];
    bool moved = false;  // wave-uniform
    float c_t = 0.f;
    if constexpr (GATE) {
        moved = a.moved[qb] != 0;
        c_t = a.centre[qb * 128u + min(threadIdx.x, C::DP - 1u)];  // (written to LDS once the rows are on their way)
    }
    // The queries' lo halves stay in LDS where registers are short (held there,
    // the sample's kernel of 97 to 128 dimensions spilled 5 to 8, with scalar row loads 46).
    constexpr bool QL_LDS = QW == 2;
    __shared__ alignas(16) _Float16 s_ql[QL_LDS ? C::QB * C::RS : 8];
    using Gate = TkGateLds<GATE ? C::QB : 1, GATE ? C::WAVES : 1>;
    __shared__ Gate G;
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t rg = wave % C::RG, qg = wave / C::RG;
    const uint32_t h = lane >> 5, j = lane & 31u;
    const uint32_t lq0 = qg * 32u * QW;  // the wave's first query within the workgroup
    const uint32_t q0 = qb * C::QB + lq0;
    const bool busy = q0 < a.n_q;  // wave-uniform

    // Tile t's rows are in set t & 1 of pre, with their ids.
    float pre[2][C::P][C::V];
    uint32_t id[2][C::P], nid[C::P];
    tk_est_ids<C, SEL, !GATE>(a, sp, tile_r0(0), id[0]);
    tk_est_ids<C, SEL, !GATE>(a, sp, tile_r0(1), id[1]);
    tk_est_rows<C, VEC>(a, id[0], pre[0]);
    tk_est_ids<C, SEL, !GATE>(a, sp, tile_r0(2), nid);
    tk_est_rows<C, VEC>(a, id[1], pre[1]);
    // Rows of tile t (0 past the last tile).
    auto tile_rows = [&](uint32_t t) -> uint32_t {
        const uint64_t r0 = tile_r0(t);
        return t < n_tiles && r0 < sp.n ? static_cast<uint32_t>(std::min<uint64_t>(sp.n - r0, C::T)) : 0u;
    };

    // A operand: the wave's queries, split, positions 16 s + 8 h .. + 7 a lane.
    f16x8 qh[QW][KS], ql[QL_LDS ? 1 : QW][QL_LDS ? 1 : KS];
    float vw[QW], vc[QW];  // the rank-2 product's query factors: sq (lanes 0-31), (gate - |q|^2) sq / 2 (lanes 32-63)
#pragma unroll
    for (int f = 0; f < QW; ++f) {
        const uint32_t q = q0 + 32u * f + j;
        const float* src = a.queries + static_cast<size_t>(q < a.n_q ? q : 0u) * a.dim;
        const bool ok = q < a.n_q;
        float x[8 * KS];
        if (a.qvec) {
#pragma unroll
            for (int e = 0; e < 8 * KS; e += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(src + min(tk_est_dim<C::DP>(2u * (e / 8) + h, e % 8), a.dim - 4u));
                x[e] = v.x, x[e + 1] = v.y, x[e + 2] = v.z, x[e + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8 * KS; ++e) x[e] = src[min(tk_est_dim<C::DP>(2u * (e / 8) + h, e % 8), a.dim - 1u)];
        }
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8 * KS; ++e) {
            x[e] = ok && tk_est_dim<C::DP>(2u * (e / 8) + h, e % 8) < a.dim ? x[e] : 0.f;
            ss += x[e] * x[e];
        }
        ss += __shfl_xor(ss, 32, 64);
        float inv;
        bool odd;
        const float sq = tk_scale(ss, inv, odd);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            f16x8 l8;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                f16x2 hi, lo;
                tk_split(odd ? 0.f : x[8 * s + e] * sq, odd ? 0.f : x[8 * s + e + 1] * sq, hi, lo);
                qh[f][s][e] = hi.x, qh[f][s][e + 1] = hi.y;
                l8[e] = lo.x, l8[e + 1] = lo.y;
            }
            if constexpr (QL_LDS) {
                if (rg == 0) *reinterpret_cast<f16x8*>(&s_ql[(lq0 + 32u * f + j) * C::RS + 16u * s + 8u * h]) = l8;
            } else {
                ql[f][s] = l8;
            }
        }
        const float gate = GATE && ok ? a.gate_at[q] : 0.f;  // (-inf: the list path answers the query, and no row passes)
        const bool pass = (odd && gate > -__builtin_inff()) || !(gate < __builtin_inff());  // every row is a candidate
        const float qgn = (1.f - TK_EST_ERR) * ss;
        vw[f] = h == 0 ? (ok ? sq : 0.f) : !ok ? -__builtin_inff() : pass ? __builtin_inff() : 0.5f * (gate - qgn) * sq;
        vc[f] = h == 0 || !ok || pass ? vw[f] : 0.5f * (gate - qgn * TK_COARSE) * sq;
        if (rg == 0 && h == 0) {
            s_isq[lq0 + 32u * f + j] = inv;
            if (GATE) {
                G.gq[lq0 + 32u * f + j] = make_float2(pass ? -__builtin_inff() : gate - TK_GATE_ROUND * gate, 2.f * inv);
                G.cnt[lq0 + 32u * f + j] =
                    stage == 2 ? a.cand_n[static_cast<size_t>(chunk) * a.q_rows + q] : 0u;
            }
        }
    }
    auto move = [&](float (&x)[C::P][C::V], const float* c) {  // one uniform branch a tile
        if (!moved) return;
#pragma unroll
        for (int e = 0; e < C::V; e += 4) {
            const f32x4 m = *reinterpret_cast<const f32x4*>(c + tk_est_col<C>(e));
#pragma unroll
            for (int p = 0; p < C::P; ++p)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[p][e + i] -= m[i];
        }
    };
    if constexpr (GATE) {
        if (threadIdx.x < C::DP) s_centre[threadIdx.x] = c_t;
        move(pre[0], a.centre + qb * 128u);
    }
    TkSplit<C, VEC> split;
    {
        const uint32_t valid = tile_rows(0);
#pragma unroll
        for (int i = 0; i < TkSplit<C, VEC>::PIECES; ++i) split.piece(i, T0, pre[0], id[0], valid, a.dim);
    }
    __syncthreads();

    auto lo_half = [&](int f, int s) -> f16x8 {  // of query fragment f, step s
        if constexpr (QL_LDS) return *reinterpret_cast<const f16x8*>(&s_ql[(lq0 + 32u * f + j) * C::RS + 16u * s + 8u * h]);
        else return ql[f][s];
    };

    // The workgroup's lists (TK_SCRATCH bounds them: 32-bit offsets).
    uint2* cand = GATE ? a.cand + (static_cast<size_t>(chunk) * a.n_q + qb * C::QB) * a.cap : nullptr;
    uint32_t held = 0;  // candidates in the wave's buffer (uniform)
    auto drain = [&]() {
        wave_lds_fence();
        for (uint32_t i = lane; i < held; i += 64) {
            const uint32_t lq = G.lq[wave][i];
            const uint32_t slot = atomicAdd(&G.cnt[lq], 1u);
            if (slot < a.cap) cand[lq * a.cap + slot] = G.buf[wave][i];
        }
        wave_lds_fence();
        held = 0;
    };
    // Tile t (in LDS buffer b = t & 1): tile t + 3's ids and tile t + 2's rows
    // are issued first; tile t + 1, loaded during tile t - 1, is split into the
    // other buffer between tile t's MFMAs.  Past the last tile the loads repeat
    // valid rows that nothing reads.
    auto tile = [&](uint32_t t, auto bc) {
        constexpr int b = decltype(bc)::value;
#pragma unroll
        for (int p = 0; p < C::P; ++p) id[b][p] = nid[p];
        tk_est_ids<C, SEL, !GATE>(a, sp, tile_r0(t + 3), nid);  // (first: the next tile's wait for them leaves the rows)
        tk_est_rows<C, VEC>(a, id[b], pre[b]);
        const uint32_t next = tile_rows(t + 1);
        if constexpr (GATE) move(pre[b ^ 1], s_centre);
        auto& B = b == 0 ? T0 : T1;
        auto& N = b == 0 ? T1 : T0;
        if (!busy) {
#pragma unroll
            for (int i = 0; i < TkSplit<C, VEC>::PIECES; ++i) split.piece(i, N, pre[b ^ 1], id[b ^ 1], next, a.dim);
        } else {
            f32x16 acc[QW];
            const TkRow* R = &B.row[rg * 32u + j];
            const float uz = h == 0 ? R->u : R->z;
#pragma unroll
            for (int f = 0; f < QW; ++f) acc[f] = f32x16{};
            const _Float16* H = &B.hi[(rg * 32u + j) * C::RS + 8u * h];
            const _Float16* W = &B.lo[(rg * 32u + j) * C::RS + 8u * h];
            // The products, each QW MFMAs and a share of the next tile's split:
            // candidates first need hi.hi only; estimates need all three, hi.hi
            // last for few dimensions (its larger sums are then rounded fewer
            // times), the three of a step together for many (which reads the
            // row's halves once).
            constexpr bool CROSS_FIRST = KS <= 4;
            constexpr int PRODUCTS = GATE ? KS : 3 * KS;
            f16x8 xh[!GATE && CROSS_FIRST ? KS : 1], xl;
            int piece = 0;
#pragma unroll
            for (int i = 0; i < PRODUCTS; ++i) {
                const bool last = !GATE && CROSS_FIRST && i >= 2 * KS;
                const int s = GATE ? i : CROSS_FIRST ? (last ? i - 2 * KS : i / 2) : i / 3;
                const int what = GATE || last ? 0 : CROSS_FIRST ? 1 + i % 2 : i % 3;  // hi.hi, lo.hi, hi.lo
                f16x8& x = xh[!GATE && CROSS_FIRST ? s : 0];
                f16x8 l8[QW];
                if (what == 1) {
#pragma unroll
                    for (int f = 0; f < QW; ++f) l8[f] = lo_half(f, s);
                }
                if (GATE || (!last && (CROSS_FIRST ? i % 2 : i % 3) == 0)) {
                    x = *reinterpret_cast<const f16x8*>(H + 16 * s);
                    if (!GATE) xl = *reinterpret_cast<const f16x8*>(W + 16 * s);
                }
#pragma unroll
                for (int f = 0; f < QW; ++f)
                    acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(what == 1 ? l8[f] : qh[f][s],
                                                                     what == 2 ? xl : x, acc[f], 0, 0, 0);
                const int end = (i + 1) * TkSplit<C, VEC>::PIECES / PRODUCTS;
#pragma unroll
                for (int k = piece; k < end; ++k) split.piece(k, N, pre[b ^ 1], id[b ^ 1], next, a.dim);
                piece = end;
                if (QW == 2) __builtin_amdgcn_sched_barrier(0);  // (up to 64 queries wait for rows, not for this order)
            }
            if constexpr (!GATE) {
#pragma unroll
                for (int f = 0; f < QW; ++f) acc[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(vw[f], uz, acc[f], 0, 0, 0);
            }
            // Register r of fragment f: query 32 f + 8 (r / 4) + 4 h + r % 4,
            // row j of the row group.
            if constexpr (GATE) {
                // hi.hi is within TK_COARSE_ERR of q.x: most fragments hold no pair
                // that could pass, whatever the cross products are.
                const float uc = h == 0 ? R->u * TK_COARSE : R->z;
                f32x16 c[QW];
#pragma unroll
                for (int f = 0; f < QW; ++f) c[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(vc[f], uc, acc[f], 0, 0, 0);
#pragma unroll
                for (int f = 0; f < QW; ++f) {
                    uint32_t mc = ~0u;  // below 2^31: a sign bit is clear (a value >= 0, or a NaN, which fails below)
#pragma unroll
                    for (int r = 0; r < 16; ++r) mc = min(mc, __float_as_uint(c[f][r]));
                    if (!__ballot(mc < 0x80000000u)) continue;
                    f32x16 cross = {};
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        const f16x8 x = *reinterpret_cast<const f16x8*>(H + 16 * s);
                        const f16x8 y = *reinterpret_cast<const f16x8*>(W + 16 * s);
                        cross = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo_half(f, s), x, cross, 0, 0, 0);
                        cross = __builtin_amdgcn_mfma_f32_32x32x16_f16(qh[f][s], y, cross, 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[f][r] += cross[r];
                    acc[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(vw[f], uz, acc[f], 0, 0, 0);
                    float m[4];
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        m[g] = fmaxf(fmaxf(fmaxf(acc[f][4 * g], acc[f][4 * g + 1]), acc[f][4 * g + 2]), acc[f][4 * g + 3]);
                    if (__ballot(fmaxf(fmaxf(fmaxf(m[0], m[1]), m[2]), m[3]) >= 0.f)) {
                        uint32_t lq = lq0 + 32u * f + 4u * h;
                        asm volatile("" : "+v"(lq));  // keeps the 32 queries' addresses out of the tile loop's registers
                        const float isx = R->isx;
                        const uint32_t row_id = R->id;
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            if (!__ballot(m[g] >= 0.f)) continue;
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                const float x = acc[f][4 * g + c];
                                const uint64_t pass = __ballot(x >= 0.f);
                                if (!pass) continue;
                                if (held > Gate::WB - 64u) drain();
                                if (x >= 0.f) {
                                    const float2 gq = G.gq[lq + 8 * g + c];
                                    const uint32_t at = held + static_cast<uint32_t>(__popcll(pass & lanemask_lt()));
                                    G.buf[wave][at] = make_uint2(__float_as_uint(gq.x - x * isx * gq.y), row_id);
                                    G.lq[wave][at] = static_cast<uint16_t>(lq + 8 * g + c);
                                }
                                held += static_cast<uint32_t>(__popcll(pass));
                            }
                        }
                    }
                }
            } else {
                const uint64_t r0 = tile_r0(t) + rg * 32u;
                const float nisx2 = -2.f * R->isx;
                if (r0 + j < sp.n) {
#pragma unroll
                    for (int f = 0; f < QW; ++f)
#pragma unroll
                        for (int r4 = 0; r4 < 4; ++r4) {
                            const uint32_t lq = lq0 + 32u * f + 8u * r4 + 4u * h;
                            const float4 iq = *reinterpret_cast<const float4*>(&s_isq[lq]);
                            float* dst = a.pd + static_cast<size_t>(qb * C::QB + lq) * a.pd_stride + r0 + j;
                            dst[0] = acc[f][4 * r4 + 0] * nisx2 * iq.x;
                            dst[a.pd_stride] = acc[f][4 * r4 + 1] * nisx2 * iq.y;
                            dst[2 * static_cast<size_t>(a.pd_stride)] = acc[f][4 * r4 + 2] * nisx2 * iq.z;
                            dst[3 * static_cast<size_t>(a.pd_stride)] = acc[f][4 * r4 + 3] * nisx2 * iq.w;
                        }
                }
            }
        }
        __syncthreads();
    };
    for (uint32_t t = 0; t < n_tiles; t += 2) {
        tile(t, std::integral_constant<int, 0>{});
        if (t + 1 < n_tiles) tile(t + 1, std::integral_constant<int, 1>{});
    }
    if constexpr (GATE) {
        drain();
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < C::QB; i += C::NT)
            a.cand_n[static_cast<size_t>(chunk) * a.q_rows + qb * C::QB + i] = G.cnt[i];
    }
}

// ---- 3. selection: one workgroup per query --------------------------------------
// An estimate L is a lower bound of its row's fp32 distance d, and
// d <= L + 3 E (|q|^2 + |x|^2) with |x|^2 <= 2 |q|^2 + 2 d, so the k rows of
// smallest L have d <= (Lk + 9.1 E |q|^2) (1 + 7 E): at least k rows lie at or
// below that bound, and every row of the answer (ties included) has its L there.
// Lk is taken from a histogram of the estimates, as the upper edge of the bin
// that holds the k-th smallest (rounded up), which only loosens the bound.
//   TK_SEL_KEPT  after the estimates: a small set's answer, or from a larger
//                one's sample the gate of its candidates (tau)
//   TK_SEL_BOUND a tighter gate from the candidates of stage 1
//   TK_SEL_CAND  the answer from the candidate lists
enum { TK_SEL_KEPT, TK_SEL_BOUND, TK_SEL_CAND };
constexpr int TK_SEL_NT = 512;
constexpr int TK_SEL_W = TK_SEL_NT / 64;
constexpr uint32_t TK_SEL_BINS = 1024;
constexpr uint32_t TK_SEL_CB = 2048;   // candidates per batch
constexpr uint32_t TK_SEL_RANK = 512;  // ... ranked by counting (one a thread) up to here, sorted above
// 16-byte loads a thread that hold `rows` kept estimates
constexpr int tk_sel_v(uint32_t rows) { return static_cast<int>(rows / (4 * TK_SEL_NT)); }
constexpr uint32_t TK_SEL_LISTS = 512;  // candidate lists a query has at most
// Candidates from which a query's selection is split: 64 queries among 300K rows,
// four of them so far away that every row is a candidate, 7730 us without,
// 958 us with; below, the parts' start and merge would be most of it.
constexpr uint32_t TK_SEL_SPLIT = 16384;
// The share of the sample in the gate from which a query goes to the list path.
// 1024 queries in ten modes, as candidates / from 1/20 on / 1/50 / 1/100: 300K rows,
// modes 30 deviations apart 562, 569, 559, 1385 us; 60 apart 2546, 1810, 1495, 1355;
// 100 apart 2945, 1447, 1447, 1446.
constexpr float TK_SEL_LIST = 1.f / 50;
constexpr int TK_SEL_ROUNDS = 4;        // histograms beyond the first
constexpr uint64_t TK_NOKEY = ~0ull;    // no candidate: after every (distance, id) key
// The largest limit that cr_topk_set_small_limit records (any from the last of TK_KEEP_MAX on is no limit).
constexpr uint32_t TK_SMALL = 1u << 18;
std::atomic<uint32_t> g_topk_small{TK_SMALL};

// Candidates are found about a common point of a query block, which leaves
// distances as they are and brings the norms, and with them the estimates'
// margins, from the distance to the origin down to the spread of the vectors.  The
// point is, dimension by dimension, the median of nine of the block's queries (a
// few far ones do not move it), or the origin where that is nearer than a quarter
// of the width of the middle ones of the nine.  A difference of two floats is
// rounded at its own size, 2.4e-7 of |q|^2 + |x|^2 in a distance: TK_EST_ERR
// holds.  The sample's selection computes it; it costs calls that need none 1 us
// there and in the candidate kernels' start.  128 dimensions, every coordinate
// moved by 100, 2M rows: 64 queries 58.4 ms without, 256 us with, 1024 queries 31.6
// ms and 1125 us.  (Kept and sampled estimates stay about the origin: it would
// be 1 to 2 us of calls of 20, and few of those rows get their distance taken.)
struct TkCentre {
    float v[9];
    float med;

    // Nine queries' dimension t (t < 128; past dim the one that stands in for it).
    __device__ __forceinline__ void load(const TkArgs& a, uint32_t q)
    {
        const uint32_t t = threadIdx.x, q0 = q / a.est_qb * a.est_qb, n = min(a.est_qb, a.n_q - q0);
        const uint32_t d = t < a.dim ? t : a.vec ? a.dim - 4u + (t & 3u) : a.dim - 1u;
        if (t < 128) {
#pragma unroll
            for (uint32_t i = 0; i < 9; ++i) v[i] = a.queries[static_cast<size_t>(q0 + i * n / 9u) * a.dim + d];
        }
    }

    // The median, and in red[0, 4) and red[4, 8) the parts of the squared sums of it and of the width.
    __device__ __forceinline__ void median(const TkArgs& a, float* red)
    {
        const uint32_t t = threadIdx.x;
        if (t >= 128) return;
        float lo[3], mid[3], hi[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            float x[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) x[j] = fabsf(v[3 * i + j]) <= 0x1p30f ? v[3 * i + j] : 0.f;
            lo[i] = fminf(fminf(x[0], x[1]), x[2]);
            hi[i] = fmaxf(fmaxf(x[0], x[1]), x[2]);
            mid[i] = __builtin_amdgcn_fmed3f(x[0], x[1], x[2]);
        }
        med = __builtin_amdgcn_fmed3f(fmaxf(fmaxf(lo[0], lo[1]), lo[2]), __builtin_amdgcn_fmed3f(mid[0], mid[1], mid[2]),
                                      fminf(fminf(hi[0], hi[1]), hi[2]));
        const float w = __builtin_amdgcn_fmed3f(hi[0], hi[1], hi[2]) - __builtin_amdgcn_fmed3f(lo[0], lo[1], lo[2]);
        const float c2 = tk_group_sum<32>(t < a.dim ? med * med : 0.f), w2 = tk_group_sum<32>(t < a.dim ? w * w : 0.f);
        if ((t & 31u) == 31u) red[t >> 5] = c2, red[4 + (t >> 5)] = w2;
    }

    // After a barrier: query q about the centre, and the block's by its first query.
    __device__ __forceinline__ void write(const TkArgs& a, uint32_t q, const float* red, const float* qv, float* qc)
    {
        const uint32_t t = threadIdx.x;
        if (t >= 128) return;
        const bool moved = red[0] + red[1] + red[2] + red[3] > 0.0625f * (red[4] + red[5] + red[6] + red[7]);
        const float c = moved ? med : 0.f;
        const float x = qv[t] - c;
        qc[t] = t < a.dim ? x : 0.f;
        if (t < a.dim) a.qc[static_cast<size_t>(q) * a.dim + t] = x;
        if (q % a.est_qb) return;
        a.centre[q / a.est_qb * 128u + t] = c;
        if (t == 0) a.moved[q / a.est_qb] = moved ? 1u : 0u;
    }
};

struct TkSelLds {
    uint64_t key[TK_SEL_CB];      // a batch: ids (or rows), then distance bits << 32 | id
    uint64_t best[2][TK_KMAX];    // the running best k, ascending (two planes)
    uint32_t hist[TK_SEL_BINS];
    uint32_t off[TK_SEL_LISTS + 1];
    float qv[128];
    float qc[128];  // the query about its block's centre (where candidates are found)
    uint32_t lds[TK_SEL_W];
    float redf[2][TK_SEL_W];
    float redc[8];
    uint32_t bin, upto, n;
};

__device__ __forceinline__ bool tk_finite(float v) { return v > -__builtin_inff() && v < __builtin_inff(); }

// Block-wide minimum of lo and maximum of hi.
__device__ __forceinline__ void tk_block_range(TkSelLds& L, float& lo, float& hi)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, o, 64));
        hi = fmaxf(hi, __shfl_xor(hi, o, 64));
    }
    if (__lane_id() == 0) L.redf[0][threadIdx.x >> 6] = lo, L.redf[1][threadIdx.x >> 6] = hi;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < TK_SEL_W; ++w) lo = fminf(lo, L.redf[0][w]), hi = fmaxf(hi, L.redf[1][w]);
}

__device__ __forceinline__ uint32_t tk_bin(float v, float lo, float scale)
{
    const float f = (v - lo) * scale;
    return f >= static_cast<float>(TK_SEL_BINS - 1) ? TK_SEL_BINS - 1 : static_cast<uint32_t>(fmaxf(f, 0.f));
}

// The bin of the k-th smallest of the binned values (TK_NOID with fewer), and
// how many values the bins up to it hold.  Every bin's count becomes that of the
// bins up to it.
__device__ __forceinline__ uint32_t tk_hist_kth(TkSelLds& L, uint32_t k, uint32_t& upto)
{
    const uint32_t t = threadIdx.x;
    static_assert(TK_SEL_BINS == 2 * TK_SEL_NT, "two bins a thread");
    if (t == 0) L.bin = TK_NOID, L.upto = 0;
    __syncthreads();  // the counts are complete
    const uint32_t h0 = L.hist[2 * t], h1 = L.hist[2 * t + 1];
    uint32_t total;
    const uint32_t e = block_excl_scan<TK_SEL_NT>(h0 + h1, L.lds, total);
    if (e < k && e + h0 + h1 >= k) {
        const bool first = e + h0 >= k;
        L.bin = 2 * t + (first ? 0u : 1u);
        L.upto = e + h0 + (first ? 0u : h1);
    }
    L.hist[2 * t] = e + h0, L.hist[2 * t + 1] = e + h0 + h1;
    __syncthreads();
    upto = L.upto;
    return L.bin;
}

// A bin's upper edge, rounded up.
__device__ __forceinline__ float tk_edge(uint32_t bin, float lo, float hi)
{
    if (bin == TK_NOID) return __builtin_inff();
    const float edge = bin == TK_SEL_BINS - 1 ? hi : lo + static_cast<float>(bin + 1) * ((hi - lo) * (1.f / TK_SEL_BINS));
    return fminf(hi, edge + 0x1p-20f * (fabsf(lo) + fabsf(hi)));
}

template <int MODE, int V>
__global__ __launch_bounds__(TK_SEL_NT) void tk_select(TkArgs a, float* out_d, int64_t* out_id)
{
    __shared__ TkSelLds L;
    const uint64_t n_rows = tk_rows(a);
    const bool small = n_rows <= a.keep;
    const uint32_t q = MODE == TK_SEL_CAND ? blockIdx.x % a.n_q : blockIdx.x;
    const uint32_t share = MODE == TK_SEL_CAND ? blockIdx.x / a.n_q : 0u;  // of the query's workgroups
    const uint32_t t = threadIdx.x;
    if (MODE != TK_SEL_KEPT && small) return;
    // More rows than kept with no candidate kernels launched, or lists that
    // overflowed with no list path launched: only a filter whose recorded
    // cardinality understates its set does that, and every row is then a
    // candidate (exact, slower; no estimate is read).
    bool all_rows = MODE == TK_SEL_KEPT && !small && a.cand_off;
    // (More than TK_KEEP rows are kept only where they are all there are.)
    const bool bound_only = MODE == TK_SEL_BOUND || (MODE == TK_SEL_KEPT && V == tk_sel_v(TK_KEEP) && !small && !all_rows);
    for (uint32_t c = t; c < 128; c += TK_SEL_NT) {
        const size_t at = static_cast<size_t>(q) * a.dim + c;
        L.qv[c] = c < a.dim ? a.queries[at] : 0.f;
        if (MODE != TK_SEL_KEPT) L.qc[c] = c < a.dim ? a.qc[at] : 0.f;
    }
    for (uint32_t i = t; i < TK_SEL_BINS; i += TK_SEL_NT) L.hist[i] = 0;
    if (t == 0) L.n = 0;
    __syncthreads();
    float qn = 0.f;  // |q|^2 as the estimates have it, each wave by itself
    {
        const float* v = MODE == TK_SEL_KEPT ? L.qv : L.qc;
        const float x = v[t & 63u], y = v[64u + (t & 63u)];
        qn = x * x + y * y;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) qn += __shfl_xor(qn, o, 64);
    }

    // The estimates: a small set's or the sample's in registers, the
    // candidate lists' through the running counts.
    const uint32_t S = MODE == TK_SEL_KEPT ? static_cast<uint32_t>(small || n_rows < a.sample ? n_rows : a.sample) : 0u;
    float4 v[V];
    uint32_t from = 0, C = 0;  // the workgroup's candidates in the lists: [from, C)
    bool split = false;      // the query has other workgroups
    const uint2* lists = a.cand + static_cast<size_t>(q) * a.cap;
    const size_t list_step = static_cast<size_t>(a.n_q) * a.cap;
    float lo = __builtin_inff(), hi = -__builtin_inff();
    auto load = [&]() {
        const float* row = a.pd + static_cast<size_t>(q) * a.pd_stride;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const uint32_t r = 4u * (t + i * TK_SEL_NT);
            v[i] = make_float4(__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""));
            if (!all_rows && r < S) {  // the row holds whole vectors
                v[i] = *reinterpret_cast<const float4*>(row + r);
                if (r + 1 >= S) v[i].y = __builtin_nanf("");
                if (r + 2 >= S) v[i].z = __builtin_nanf("");
                if (r + 3 >= S) v[i].w = __builtin_nanf("");
            }
        }
    };
    TkCentre centre;
    if constexpr (MODE == TK_SEL_KEPT) {
        if (bound_only) centre.load(a, q);
        load();
        if (bound_only) centre.median(a, L.redc);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const float e[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (tk_finite(e[c])) lo = fminf(lo, e[c]), hi = fmaxf(hi, e[c]);
        }
    } else {
        const bool lists = !a.list_off && a.q_over[q];  // (nothing wrote its counts)
        if (MODE == TK_SEL_BOUND && lists) return;
        uint32_t n = t < a.n_cw && !lists ? a.cand_n[static_cast<size_t>(t) * a.q_rows + q] : 0u;
        const bool over = __syncthreads_or(n > a.cap) || lists;
        n = min(n, a.cap);
        const uint32_t e = block_excl_scan<TK_SEL_NT>(n, L.lds, C);
        L.off[t] = e;
        if (t == 0) L.off[TK_SEL_LISTS] = C;
        __syncthreads();
        if constexpr (MODE == TK_SEL_CAND) {
            split = a.parts > 1 && C > TK_SEL_SPLIT && !over;
            if (share > 0 && !split) return;
            if (split) {
                from = static_cast<uint32_t>(static_cast<uint64_t>(C) * share / a.parts);
                C = static_cast<uint32_t>(static_cast<uint64_t>(C) * (share + 1) / a.parts);
            }
            if (!a.list_off) {
                if (t == 0) {
                    a.q_over[q] = over ? 1u : 0u;
                    if (over) a.qb_over[q / TK_QB] = 1u;
                }
                if (over)  // the list path answers: its state (the gate stays its bound)
                    for (uint32_t c = t; c < a.n_chunks; c += TK_SEL_NT)
                        a.tau_m[static_cast<size_t>(c) * a.n_q + q] = 0x7F800000u;
                if (over) return;
            } else {
                all_rows = over;
            }
        }
    }
    auto cand_at = [&](uint32_t i) -> uint2 {  // candidate i of the query's lists
        uint32_t c = 0;
#pragma unroll
        for (uint32_t step = TK_SEL_LISTS / 2; step > 0; step >>= 1)
            if (L.off[c + step] <= i) c += step;
        return lists[c * list_step + (i - L.off[c])];
    };
    if constexpr (MODE != TK_SEL_KEPT) {
        for (uint32_t i = from + t; i < C; i += TK_SEL_NT) {
            const float e = __uint_as_float(cand_at(i).x);
            if (tk_finite(e)) lo = fminf(lo, e), hi = fmaxf(hi, e);
        }
    }
    tk_block_range(L, lo, hi);
    if (MODE == TK_SEL_KEPT && bound_only) centre.write(a, q, L.redc, L.qv, L.qc);
    float scale = hi > lo ? static_cast<float>(TK_SEL_BINS) / (hi - lo) : 0.f;
    if constexpr (MODE == TK_SEL_KEPT) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const float e[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (tk_finite(e[c])) atomicAdd(&L.hist[tk_bin(e[c], lo, scale)], 1u);
        }
    } else {
        for (uint32_t i = from + t; i < C; i += TK_SEL_NT) {
            const float e = __uint_as_float(cand_at(i).x);
            if (tk_finite(e)) atomicAdd(&L.hist[tk_bin(e, lo, scale)], 1u);
        }
    }
    uint32_t upto;
    uint32_t bin = tk_hist_kth(L, a.k, upto);
    float edge = tk_edge(bin, lo, hi);
    // A few far values stretch the range until one bin holds nearly every other:
    // again over the k-th value's bin alone (lower ones count in its first bin),
    // with the estimates from memory, where they came from (little code: its
    // instructions are fetched on every call; unrolled over the registers it
    // cost calls that never come here 1.5 us).  One row in 2000 at 1000 times the
    // others' size, 300K rows, 64 queries: 1362 us without, 102 with.
    const uint32_t few = max(4 * a.k + 256u, bound_only ? 0u : TK_SEL_RANK);
    bool again = false;
    for (int round = 0; round < TK_SEL_ROUNDS && upto > few && edge < hi; ++round) {
        lo = fmaxf(lo, lo + static_cast<float>(bin) * ((hi - lo) * (1.f / TK_SEL_BINS)) - 0x1p-20f * (fabsf(lo) + fabsf(hi)));
        hi = edge;
        for (uint32_t i = t; i < TK_SEL_BINS; i += TK_SEL_NT) L.hist[i] = 0;
        __syncthreads();
        scale = hi > lo ? static_cast<float>(TK_SEL_BINS) / (hi - lo) : 0.f;
        again = true;
#pragma unroll 4
        for (uint32_t i = from + t; i < (MODE == TK_SEL_KEPT ? S : C); i += TK_SEL_NT) {
            const float e = MODE == TK_SEL_KEPT ? a.pd[static_cast<size_t>(q) * a.pd_stride + i] : __uint_as_float(cand_at(i).x);
            if (tk_finite(e) && e <= hi) atomicAdd(&L.hist[tk_bin(e, lo, scale)], 1u);
        }
        bin = tk_hist_kth(L, a.k, upto);
        edge = tk_edge(bin, lo, hi);
    }
    // Candidate estimates were rounded down by up to twice TK_GATE_ROUND of the
    // gate that they passed, the first candidates' being the largest.
    const float gate = MODE == TK_SEL_KEPT ? 0.f : __uint_as_float(a.tau_first[q]);
    float bound = edge;
    if (bound < __builtin_inff())
        bound = fmaxf(bound + 9.1f * TK_EST_ERR * qn + 2.f * TK_GATE_ROUND * gate, 0.f) * (1.f + 8.f * TK_EST_ERR);
    // The margin is of the size of the norms: on vectors far from the origin it
    // lets many through.  The rows with the k-th smallest estimates are the
    // nearest all the same (an estimate's error is far below its bound), so
    // their distances are taken first, and their k-th bounds the answer.  128
    // dimensions, every coordinate moved by 20 and by 40 (|q|^2 at 317 and 1182
    // times d_k): 10000 rows, 1024 queries 116 -> 81 us and 281 -> 110, 2M rows
    // 3590 -> 1790 and 15.4 -> 3.6 ms.
    const bool near_first = MODE != TK_SEL_BOUND && !all_rows && bound < __builtin_inff() &&
                            ((again && bound > hi) || L.hist[tk_bin(bound, lo, scale)] > (bound_only ? 2 * a.k + 32u : few));
    auto write_bound = [&](bool lists) {
        if (t == 0) {
            if (MODE == TK_SEL_KEPT) a.q_over[q] = lists ? 1u : 0u;
            const float at = MODE == TK_SEL_KEPT ? bound : fminf(bound, gate);
            a.tau[q] = __float_as_uint(at);
            a.gate_at[q] = lists ? -__builtin_inff() : at;
            if (MODE == TK_SEL_KEPT) a.tau_first[q] = __float_as_uint(bound), a.part_done[q] = 0;
            if (MODE == TK_SEL_KEPT && !a.list_off && q % TK_QB == 0) a.qb_over[q / TK_QB] = 0;
        }
    };
    if (bound_only && !near_first) {
        write_bound(false);
        return;
    }
    if (all_rows) bound = __builtin_inff();

    // Candidates in batches: fp32 direct distances, an order by (distance, id),
    // and a merge into the running best k.
    uint32_t nb = 0, cur = 0;
    auto sort = [&](uint32_t n) {  // key[0, n), ascending
        uint32_t P = 2;
        while (P < n) P <<= 1;
        for (uint32_t i = n + t; i < P; i += TK_SEL_NT) L.key[i] = TK_NOKEY;
        __syncthreads();
        for (uint32_t size = 2; size <= P; size <<= 1) {
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                for (uint32_t i = t; i < P / 2; i += TK_SEL_NT) {
                    const uint32_t l = 2 * i - (i & (stride - 1));
                    const uint64_t x = L.key[l], y = L.key[l + stride];
                    if ((y < x) == ((l & size) == 0)) L.key[l] = y, L.key[l + stride] = x;
                }
                __syncthreads();
            }
        }
    };
    auto flush = [&](uint32_t nbatch, bool rows) {  // the batch's ids (or rows of the set) are in key
        for (uint32_t c0 = 0; c0 < nbatch; c0 += TK_SEL_NT / 8) {  // eight threads (of one wave) per candidate
            const uint32_t c = c0 + t / 8, part = t % 8;
            float e2 = 0.f;
            uint32_t id = 0;
            if (c < nbatch) {
                id = static_cast<uint32_t>(L.key[c]);
                if (rows && a.sel) id = a.sel[id];
                // the part's 16 dimensions, all loaded before any is used (zeros
                // past dim, where qv is zero too, add nothing)
                const float* x = a.base + static_cast<size_t>(id) * a.dim + part * 16;
#pragma unroll
                for (uint32_t hh = 0; hh < 16; hh += 8) {  // two halves of 8
                    float xv[8];
                    if (a.vec) {  // dim % 4 == 0, 16-byte aligned rows
#pragma unroll
                        for (uint32_t q4 = 0; q4 < 8; q4 += 4) {
                            const float4 w = part * 16 + hh + q4 < a.dim
                                                 ? *reinterpret_cast<const float4*>(x + hh + q4)
                                                 : make_float4(0.f, 0.f, 0.f, 0.f);
                            xv[q4] = w.x, xv[q4 + 1] = w.y, xv[q4 + 2] = w.z, xv[q4 + 3] = w.w;
                        }
                    } else {
#pragma unroll
                        for (uint32_t s2 = 0; s2 < 8; ++s2) xv[s2] = part * 16 + hh + s2 < a.dim ? x[hh + s2] : 0.f;
                    }
#pragma unroll
                    for (uint32_t s2 = 0; s2 < 8; ++s2) {
                        const float e = L.qv[part * 16 + hh + s2] - xv[s2];
                        e2 = fmaf(e, e, e2);
                    }
                }
            }
            e2 += __shfl_xor(e2, 1, 64);
            e2 += __shfl_xor(e2, 2, 64);
            e2 += __shfl_xor(e2, 4, 64);
            if (c < nbatch && part == 0)  // non-negative: the bits order as values; NaN is no distance
                L.key[c] = e2 == e2 ? (static_cast<uint64_t>(__float_as_uint(e2)) << 32) | id : TK_NOKEY;
        }
        for (uint32_t i = t; i < TK_KMAX; i += TK_SEL_NT) L.best[cur ^ 1][i] = TK_NOKEY;
        const uint32_t nbt = min(nbatch, a.k);
        if (nb == 0 && nbatch <= TK_SEL_RANK) {
            // few: each thread counts the keys below its own
            __syncthreads();
            const uint64_t mine = t < nbatch ? L.key[t] : TK_NOKEY;
            uint32_t r = 0;
            if (t < nbatch)
                for (uint32_t i = 0; i < nbatch; ++i) r += L.key[i] < mine ? 1u : 0u;
            if (mine != TK_NOKEY && r < a.k) L.best[cur ^ 1][r] = mine;
        } else {
            sort(nbatch);
            // Merge: an entry's rank is its index plus the number of entries of
            // the other list before it (all keys but TK_NOKEY are distinct).
            auto below = [](const uint64_t* p, uint32_t n, uint64_t y) {
                uint32_t l = 0, r = n;
                while (l < r) {
                    const uint32_t m = (l + r) >> 1;
                    if (p[m] < y) l = m + 1;
                    else r = m;
                }
                return l;
            };
            if (t < nb) {
                const uint64_t x = L.best[cur][t];
                const uint32_t r = t + below(L.key, nbt, x);
                if (x != TK_NOKEY && r < a.k) L.best[cur ^ 1][r] = x;
            } else if (t - nb < nbt) {
                const uint64_t x = L.key[t - nb];
                const uint32_t r = t - nb + below(L.best[cur], nb, x);
                if (x != TK_NOKEY && r < a.k) L.best[cur ^ 1][r] = x;
            }
        }
        nb = min(a.k, nb + nbt);
        cur ^= 1;
        if (t == 0) L.n = 0;
        __syncthreads();
        if (nb == a.k) {  // the k-th best so far bounds the answer
            const uint64_t kth = L.best[cur][a.k - 1];
            if (kth != TK_NOKEY) bound = fminf(bound, __uint_as_float(static_cast<uint32_t>(kth >> 32)));
        }
    };
    // Slots of the batch come from an LDS counter; a batch that the next
    // TK_SEL_NT values could overflow is flushed first.
    auto room = [&]() {
        __syncthreads();  // the slots so far are taken
        const uint32_t n = L.n;
        __syncthreads();  // every thread has read the count
        if (n > TK_SEL_CB - TK_SEL_NT) flush(n, MODE == TK_SEL_KEPT || all_rows);
    };
    // Whether the list path is the better one from the start: of the sampled rows,
    // more than TK_SEL_LIST pass the candidates' gate, or so many that the lists
    // would overflow.  An estimate here lies about 2 E |q|^2 under the distance (the
    // near rows' norms are the query's), the gate's about the centre 2 E |q'|^2.
    auto too_many = [&]() -> bool {
        float x = L.qc[t & 63u], y = L.qc[64u + (t & 63u)];
        float qm = x * x + y * y;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) qm += __shfl_xor(qm, o, 64);
        const float top = bound + 2.f * TK_EST_ERR * (qm - qn);
        uint32_t n = 0;
#pragma unroll 4
        for (uint32_t i = t; i < S; i += TK_SEL_NT) n += a.pd[static_cast<size_t>(q) * a.pd_stride + i] <= top ? 1u : 0u;
        n = block_sum<TK_SEL_NT>(n, L.lds);
        return n > S * TK_SEL_LIST || static_cast<float>(n) * static_cast<float>(n_rows) > 0.7f * S * a.cap * a.n_cw;
    };
    if (__builtin_expect(near_first, 0)) {
        // The rows up to the edge, TK_SEL_CB of them where ties make them more,
        // which bound the k-th distance as well.  They are taken again below.
        if constexpr (MODE == TK_SEL_KEPT) {
            uint32_t mine = 0;
#pragma unroll
            for (int i = 0; i < V; ++i)
                mine += (v[i].x <= edge ? 1u : 0u) + (v[i].y <= edge ? 1u : 0u) + (v[i].z <= edge ? 1u : 0u) +
                        (v[i].w <= edge ? 1u : 0u);
            uint32_t total;
            uint32_t at = block_excl_scan<TK_SEL_NT>(mine, L.lds, total);
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float e[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (!(e[c] <= edge)) continue;
                    const uint32_t r = 4u * (t + i * TK_SEL_NT) + c;
                    // (a sampled row's place in the set)
                    if (at < TK_SEL_CB) L.key[at] = bound_only && S < n_rows ? (r * n_rows) >> a.sample_lg : r;
                    ++at;
                }
            }
            if (t == 0) L.n = total;
        } else {
            for (uint32_t i = from + t; i < C; i += TK_SEL_NT) {
                const uint2 e = cand_at(i);
                if (!(__uint_as_float(e.x) <= edge)) continue;
                const uint32_t at = atomicAdd(&L.n, 1u);
                if (at < TK_SEL_CB) L.key[at] = e.y;
            }
        }
        __syncthreads();
        flush(min(L.n, TK_SEL_CB), MODE == TK_SEL_KEPT);
        if (bound_only) {
            write_bound(MODE == TK_SEL_KEPT && !a.list_off && too_many());
            return;
        }
        nb = 0;
        if constexpr (MODE == TK_SEL_KEPT) load();  // (not held in registers all the while)
    }
    if (all_rows) {
        for (uint64_t r0 = 0; r0 < n_rows; r0 += TK_SEL_NT) {
            room();
            if (r0 + t < n_rows) L.key[atomicAdd(&L.n, 1u)] = r0 + t;
        }
    } else if constexpr (MODE == TK_SEL_KEPT) {
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < V; ++i)
            mine += (v[i].x <= bound ? 1u : 0u) + (v[i].y <= bound ? 1u : 0u) + (v[i].z <= bound ? 1u : 0u) +
                    (v[i].w <= bound ? 1u : 0u);
        uint32_t total;
        uint32_t at = block_excl_scan<TK_SEL_NT>(mine, L.lds, total);
        if (total <= TK_SEL_CB) {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float e[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (e[c] <= bound) L.key[at++] = 4u * (t + i * TK_SEL_NT) + c;
            }
            if (t == 0) L.n = total;
        } else {
            const float* row = a.pd + static_cast<size_t>(q) * a.pd_stride;
            for (uint32_t r0 = 0; r0 < S; r0 += TK_SEL_NT) {
                room();
                if (r0 + t < S && row[r0 + t] <= bound) L.key[atomicAdd(&L.n, 1u)] = r0 + t;
            }
        }
    } else {
        for (uint32_t i0 = from; i0 < C; i0 += TK_SEL_NT) {
            room();
            if (i0 + t < C) {
                const uint2 e = cand_at(i0 + t);
                if (__uint_as_float(e.x) <= bound) L.key[atomicAdd(&L.n, 1u)] = e.y;
            }
        }
    }
    __syncthreads();
    const uint32_t left = L.n;
    if (left) flush(left, MODE == TK_SEL_KEPT || all_rows);
    if (MODE == TK_SEL_CAND && split) {
        uint64_t* mine = a.part_key + (static_cast<size_t>(q) * a.parts + share) * a.k;
        for (uint32_t r = t; r < a.k; r += TK_SEL_NT) mine[r] = r < nb ? L.best[cur][r] : TK_NOKEY;
        __threadfence();  // each thread's keys before its workgroup's count
        __syncthreads();
        if (t == 0) L.n = atomicAdd(&a.part_done[q], 1u);
        __syncthreads();
        if (L.n != a.parts - 1u) return;
        __threadfence();
        const uint32_t n = a.parts * a.k;  // at most TK_SEL_CB
        const uint64_t* all = a.part_key + static_cast<size_t>(q) * n;
        for (uint32_t i = t; i < n; i += TK_SEL_NT)
            L.key[i] = __hip_atomic_load(all + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sort(n);  // (a barrier first)
        for (uint32_t r = t; r < a.k; r += TK_SEL_NT) L.best[cur][r] = L.key[r];
        nb = a.k;
    }
    for (uint32_t r = t; r < a.k; r += TK_SEL_NT) {
        const uint64_t x = r < nb ? L.best[cur][r] : TK_NOKEY;
        const bool ok = x != TK_NOKEY;
        out_d[static_cast<size_t>(q) * a.k + r] = ok ? __uint_as_float(static_cast<uint32_t>(x >> 32)) : __builtin_inff();
        out_id[static_cast<size_t>(q) * a.k + r] = ok ? static_cast<int64_t>(static_cast<uint32_t>(x)) : int64_t(-1);
    }
}

// The call's state (tk_init_from), when no enumeration kernel sets it.
__global__ __launch_bounds__(256) void tk_init(TkArgs a)
{
    tk_init_from(a, static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x, static_cast<uint64_t>(gridDim.x) * 256u);
}

// One launch of tk_est: n_cw workgroups a query block, rounded up to the XCDs.
template <int KS, int QW, int QG, bool GATE>
void launch_est(const TkArgs& a, uint32_t n_qb, uint32_t stage, hipStream_t s)
{
    const uint32_t grid = (a.n_cw * n_qb + 7u) / 8u * 8u;
    constexpr int NT = TkEst<KS, QW, QG>::NT;
    CR_TIMED(GATE ? "tk_gate" : "tk_pairs", s);
    if (a.sel && a.vec)
        tk_est<KS, QW, QG, true, true, GATE><<<grid, NT, 0, s>>>(a, n_qb, stage);
    else if (a.sel)
        tk_est<KS, QW, QG, true, false, GATE><<<grid, NT, 0, s>>>(a, n_qb, stage);
    else if (a.vec)
        tk_est<KS, QW, QG, false, true, GATE><<<grid, NT, 0, s>>>(a, n_qb, stage);
    else
        tk_est<KS, QW, QG, false, false, GATE><<<grid, NT, 0, s>>>(a, n_qb, stage);
}

template <int MODE, int V = 1>
int launch_select(const TkArgs& a, float* out_d, int64_t* out_ids, hipStream_t s)
{
    CR_TIMED("tk_select", s);
    tk_select<MODE, V><<<MODE == TK_SEL_CAND ? a.n_q * a.parts : a.n_q, TK_SEL_NT, 0, s>>>(a, out_d, out_ids);
    CR_LAUNCH_CHECK();
    return CR_OK;
}

// The estimate path: the answer of a small set, or the sample's bound, the
// candidates (in two stages when one bound would let too many through) and
// the answer from them.
template <int KS, int QW, int QG>
int launch_gated(const TkArgs& a, uint32_t n_qb, bool two_stages, float* out_d, int64_t* out_ids, hipStream_t s)
{
    launch_est<KS, QW, QG, false>(a, n_qb, 0, s);
    CR_LAUNCH_CHECK();
    auto* select = a.keep <= TK_KEEP          ? launch_select<TK_SEL_KEPT, tk_sel_v(TK_KEEP)>
                   : a.keep <= TK_KEEP_MAX[0] ? launch_select<TK_SEL_KEPT, tk_sel_v(TK_KEEP_MAX[0])>
                   : a.keep <= TK_KEEP_MAX[1] ? launch_select<TK_SEL_KEPT, tk_sel_v(TK_KEEP_MAX[1])>
                                              : launch_select<TK_SEL_KEPT, tk_sel_v(TK_KEEP_MAX[2])>;
    CR_RET(select(a, out_d, out_ids, s));
    if (a.cand_off) return CR_OK;
    TkArgs g = a;  // the candidates' queries are the moved ones
    g.queries = a.qc;
    g.qvec = a.dim % 4 == 0;
    if (two_stages) {
        launch_est<KS, QW, QG, true>(g, n_qb, 1, s);
        CR_LAUNCH_CHECK();
        CR_RET(launch_select<TK_SEL_BOUND>(a, out_d, out_ids, s));
    }
    launch_est<KS, QW, QG, true>(g, n_qb, two_stages ? 2 : 0, s);
    CR_LAUNCH_CHECK();
    return launch_select<TK_SEL_CAND>(a, out_d, out_ids, s);
}

template <int QW, int QG>
int launch_gated_dim(const TkArgs& a, uint32_t n_qb, bool two_stages, float* out_d, int64_t* out_ids, hipStream_t s)
{
    if (a.dim <= 32) return launch_gated<2, QW, QG>(a, n_qb, two_stages, out_d, out_ids, s);
    if (a.dim <= 64) return launch_gated<4, QW, QG>(a, n_qb, two_stages, out_d, out_ids, s);
    if (a.dim <= 96) return launch_gated<6, QW, QG>(a, n_qb, two_stages, out_d, out_ids, s);
    return launch_gated<8, QW, QG>(a, n_qb, two_stages, out_d, out_ids, s);
}

template <int DP>
int launch_dist(const TkArgs& a, uint32_t grid, hipStream_t s)
{
    CR_TIMED("tk_dist", s);
    if (a.sel)
        tk_dist<DP, true><<<grid, TK_NT, 0, s>>>(a);
    else
        tk_dist<DP, false><<<grid, TK_NT, 0, s>>>(a);
    CR_LAUNCH_CHECK();
    return CR_OK;
}

}  // namespace
}  // namespace crimpl

using namespace crimpl;

extern "C" int cr_topk_filtered(const float* d_base, uint64_t n_base, const float* d_queries, uint32_t n_q,
                                uint32_t dim, const cr_gpu_roaring* filter, uint32_t k, float* d_out_dist,
                                int64_t* d_out_ids, cr_stream_t stream)
{
    if (n_q == 0 || k == 0) return CR_OK;
    if (!d_queries || !d_out_dist || !d_out_ids || (n_base && !d_base) || dim == 0) {
        set_error("cr_topk_filtered: invalid argument");
        return CR_ERR_INVALID;
    }
    if (dim > 128 || k > TK_KMAX || n_base > 0xFFFFFFFFull) {
        set_error("cr_topk_filtered: supported up to dim 128, k %u and 2^32-1 base vectors (dim %u, k %u)", TK_KMAX,
                  dim, k);
        return CR_ERR_UNSUPPORTED;
    }
    hipStream_t s = as_stream(stream);
    const uint32_t cus = num_cus();
    const uint64_t nb = (n_base + TK_ENUM_IDS - 1) / TK_ENUM_IDS;

    TkArgs a{};
    a.base = d_base;
    a.queries = d_queries;
    a.n_base = n_base;
    a.n_q = n_q;
    a.dim = dim;
    a.k = k;
    a.vec = (dim % 4 == 0) && (reinterpret_cast<uintptr_t>(d_base) % 16 == 0);
    a.qvec = (dim % 4 == 0) && (reinterpret_cast<uintptr_t>(d_queries) % 16 == 0);

    // The most rows that can pass: a filter's recorded cardinality (the
    // library's uploads and fused multi_and record it, and the reference's
    // conversions rely on it too, src/to_csr.cu:212-216), plus one per container
    // for a multi_and's full containers stored as 65535.  An understated one
    // costs time, never the answer.
    const uint64_t rows_ub = filter && filter->total_cardinality > 0
                                 ? std::min<uint64_t>(n_base, filter->total_cardinality + filter->n_containers)
                                 : n_base;

    // Rows whose estimates are all kept: two launches over every estimate are
    // less than the sample, its bound, the candidates and the choice, as long as
    // the estimates are few.  us kept / by candidates, 128 dimensions (64 where
    // said): 65 queries, 17000 rows 26 / 46, 65000 rows 50 / 56 (64 dimensions,
    // 50000 rows 41 / 39); 300 queries, 32000 rows 60 / 71, 45000 rows 77 / 76; 700
    // queries, 24500 rows 61 / 86, 32000 rows 97 / 90.
    const uint32_t limit = g_topk_small.load();
    const uint32_t most = n_q <= 256 ? (dim > 64 ? 65536 : 40960) : n_q <= 512 ? 40960 : 24576;
    a.keep = TK_KEEP;
    for (uint32_t m : TK_KEEP_MAX)
        if (rows_ub > a.keep && rows_ub <= most && m <= most) a.keep = m;
    auto fit = [&](uint32_t q_rows) { return TK_SCRATCH / (4ull * q_rows) / TK_ROWS * TK_ROWS; };  // estimates within the scratch limit
    const uint64_t fit64 = fit((n_q + 63) / 64 * 64);
    a.keep = static_cast<uint32_t>(std::min<uint64_t>(std::min(limit, a.keep), fit64));
    a.cand_off = rows_ub <= a.keep;

    // The estimate path: 256 queries a workgroup, or 64 for the few that read
    // the rows only once anyway and for kept rows, whose tiles are too few to share
    // the queries' preparation (12000 rows: 65 queries 24.1 us with 256, 23.1 with 64;
    // 256 queries 32.3 and 28.1; 1024 queries 54.4 and 51.6).
    const bool few = n_q <= 64 || a.cand_off;
    const uint32_t est_qb = few ? 64 : 256;
    const uint32_t n_qb = (n_q + est_qb - 1) / est_qb;
    a.q_rows = n_qb * est_qb;
    a.est_qb = est_qb;
    a.n_cw = std::min<uint32_t>(TK_SEL_LISTS, std::max<uint32_t>(1, (few ? 2 : 1) * cus / n_qb));
    a.sample_lg = 14;
    static_assert(TK_KEEP == 1u << 14, "the sample is at most the kept rows");
    while ((1ull << a.sample_lg) > fit(a.q_rows) && a.sample_lg > 0) --a.sample_lg;
    a.sample = 1u << a.sample_lg;
    // limit 0 turns it off; so does a batch of queries too large for a sample
    // that bounds the k-th distance.
    a.gate = limit > 0 && a.sample >= std::max<uint32_t>(1024, 8 * k);
    if (!a.gate) a.keep = 0;
    else a.keep = static_cast<uint32_t>(std::min<uint64_t>(a.keep, fit(a.q_rows)));
    if (rows_ub > a.keep) a.keep = std::min(a.keep, TK_KEEP);
    a.pd_stride = std::max((a.keep + 63u) / 64u * 64u, a.sample);
    a.cand_off = a.gate && rows_ub <= a.keep;
    // Lists that hold every row a workgroup sees need no list path behind them.
    const uint64_t list_rows = ((rows_ub + TK_ROWS - 1) / TK_ROWS + a.n_cw - 1) / a.n_cw * TK_ROWS +
                               TK_ROWS;  // two stages may give a workgroup one tile more
    const uint64_t lists_fit = TK_SCRATCH / (8ull * n_q * a.n_cw);
    const bool whole = list_rows <= std::min<uint64_t>(lists_fit, TK_CAND_WHOLE / a.n_cw);
    // One bound from the sample lets about k rows / sample candidates a query
    // through.  A second bound, from the first 16th of the tiles, costs two
    // launches; it saves most of the lists, and of the cross products (a fragment
    // computes them for any candidate it may hold).
    const double expected = static_cast<double>(k) * static_cast<double>(rows_ub) / a.sample;
    const bool two_stages = expected > TK_TWO_STAGE || expected * n_q > TK_TWO_STAGE_ALL;
    const uint64_t many = std::max<uint64_t>(TK_CAND_MANY, static_cast<uint64_t>(8 * expected / (two_stages ? TK_STAGE : 1)));
    a.cap = static_cast<uint32_t>(whole ? list_rows : std::min<uint64_t>({TK_CAND_CAP, lists_fit, many / a.n_cw}));
    a.list_off = a.gate && (a.cand_off || whole);

    // The list path: enough (chunk, query block) workgroups to cover every CU once.
    const uint32_t list_qb = (n_q + TK_QB - 1) / TK_QB;
    uint32_t n_chunks = std::max<uint32_t>(8, (cus + list_qb - 1) / list_qb);
    n_chunks = (n_chunks + 7) / 8 * 8;
    a.n_chunks = n_chunks;
    a.m_rank = std::max<uint32_t>(1, (2 * k + n_chunks - 1) / n_chunks);

    Carver cv;
    const size_t o_counts = cv.add(filter ? nb * 4 : 0);
    const size_t o_nsel = cv.add(4);
    const size_t o_sel = cv.add(filter ? n_base * 4 : 0);
    const size_t o_tau = cv.add(static_cast<size_t>(n_q) * 4);
    const size_t lists = a.list_off ? 0 : static_cast<size_t>(n_chunks) * n_q * k;
    const size_t o_ld = cv.add(2 * lists * 4);
    const size_t o_li = cv.add(2 * lists * 4);
    const size_t o_ln = cv.add(a.list_off ? 0 : static_cast<size_t>(n_chunks) * n_q * 4);
    const size_t o_taum = cv.add(a.list_off ? 0 : static_cast<size_t>(n_chunks) * n_q * 4);
    const size_t o_pd = cv.add(a.gate ? static_cast<size_t>(a.q_rows) * a.pd_stride * 4 : 0);
    const bool cands = a.gate && !a.cand_off;
    const size_t o_cand = cv.add(cands ? static_cast<size_t>(n_q) * a.n_cw * a.cap * 8 : 0);
    const size_t o_qc = cv.add(cands ? static_cast<size_t>(n_q) * dim * 4 : 0);
    const size_t o_centre = cv.add(cands ? static_cast<size_t>(n_qb) * 128 * 4 : 0);
    const size_t o_moved = cv.add(cands ? static_cast<size_t>(n_qb) * 4 : 0);
    a.parts = n_q <= 64 ? std::max<uint32_t>(1, std::min<uint32_t>({64, 4 * cus / n_q, TK_SEL_CB / k})) : 1;
    const size_t o_pkey = cv.add(cands ? static_cast<size_t>(n_q) * a.parts * k * 8 : 0);
    const size_t o_pdone = cv.add(cands ? static_cast<size_t>(n_q) * 4 : 0);
    const size_t o_gate_at = cv.add(cands ? static_cast<size_t>(n_q) * 4 : 0);
    const size_t o_tau_first = cv.add(cands ? static_cast<size_t>(n_q) * 4 : 0);
    const size_t o_candn = cv.add(cands ? static_cast<size_t>(a.q_rows) * a.n_cw * 4 : 0);
    const size_t o_qover = cv.add(cands ? static_cast<size_t>(n_q) * 4 : 0);
    const size_t o_qbover = cv.add(cands ? static_cast<size_t>(list_qb) * 4 : 0);
    Scratch sc;
    CR_RET(sc.alloc(cv.total, s));
    a.tau = sc.at<uint32_t>(o_tau);
    a.list_d = sc.at<float>(o_ld);
    a.list_id = sc.at<uint32_t>(o_li);
    a.list_n = sc.at<uint32_t>(o_ln);
    a.plane = lists;
    a.tau_m = sc.at<uint32_t>(o_taum);
    a.pd = sc.at<float>(o_pd);
    a.cand = sc.at<uint2>(o_cand);
    a.qc = sc.at<float>(o_qc);
    a.centre = sc.at<float>(o_centre);
    a.moved = sc.at<uint32_t>(o_moved);
    a.part_key = sc.at<uint64_t>(o_pkey);
    a.part_done = sc.at<uint32_t>(o_pdone);
    a.gate_at = sc.at<float>(o_gate_at);
    a.tau_first = sc.at<uint32_t>(o_tau_first);
    a.cand_n = sc.at<uint32_t>(o_candn);
    a.q_over = sc.at<uint32_t>(o_qover);
    a.qb_over = sc.at<uint32_t>(o_qbover);

    if (!a.gate && (!filter || nb == 0)) {
        tk_init<<<static_cast<unsigned>((static_cast<uint64_t>(n_chunks) * n_q + 255) / 256), 256, 0, s>>>(a);
        CR_LAUNCH_CHECK();
    }
    if (filter) {
        cr_gpu_roaring_view cv_view;
        CR_RET(cr_make_view(filter, &cv_view));
        GpuRoaringView v;
        static_assert(sizeof(v) == sizeof(cv_view), "view layout");
        std::memcpy(&v, &cv_view, sizeof(v));
        a.sel = sc.at<uint32_t>(o_sel);
        a.n_sel = sc.at<uint32_t>(o_nsel);
        if (nb == 0) {
            CR_RET(fill_u32(sc.at<uint32_t>(o_nsel), 0u, 1, s));
        } else {
            CR_TIMED("tk_enum", s);
            tk_enum_count<<<static_cast<unsigned>(nb), TK_ENUM_NT, 0, s>>>(v, n_base, sc.at<uint32_t>(o_counts), a);
            tk_enum_write<<<static_cast<unsigned>(nb), TK_ENUM_NT, 0, s>>>(v, n_base, sc.at<uint32_t>(o_counts),
                                                                           sc.at<uint32_t>(o_sel), sc.at<uint32_t>(o_nsel));
        }
        CR_LAUNCH_CHECK();
    }
    if (a.gate) {
        const int rc = few ? launch_gated_dim<1, 2>(a, n_qb, two_stages, d_out_dist, d_out_ids, s)
                           : launch_gated_dim<2, 4>(a, n_qb, two_stages, d_out_dist, d_out_ids, s);
        CR_RET(rc);
    }
    if (!a.list_off) {
        const uint32_t grid = n_chunks * list_qb;
        if (dim <= 32) {
            CR_RET(launch_dist<32>(a, grid, s));
        } else if (dim <= 64) {
            CR_RET(launch_dist<64>(a, grid, s));
        } else {
            CR_RET(launch_dist<128>(a, grid, s));
        }
        CR_TIMED("tk_merge", s);
        tk_merge<<<(n_q + 3) / 4, TK_MERGE_NT, 0, s>>>(a, a.list_d, a.list_id, a.plane, a.list_n, n_chunks, n_q, k,
                                                        d_out_dist, d_out_ids);
        CR_LAUNCH_CHECK();
    }
    return CR_OK;
}

extern "C" uint32_t cr_topk_set_small_limit(uint32_t rows)
{
    const uint32_t prev = g_topk_small.load();
    g_topk_small.store(std::min<uint32_t>(rows, TK_SMALL));
    return prev;
}
