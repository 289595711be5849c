// upload_from_device_bitset / upload_from_bitset on gfx950.
//
// Semantics follow src/upload_ids.cu:606-893 (reference): 65536-bit chunks,
// every non-empty chunk becomes a BITMAP container (cards clamp 65536->0),
// complement when the popcount exceeds U/2 (strict), the inverted copy is
// masked only in the tail word U/32, max_key = last non-empty chunk,
// total_cardinality = the input's popcount.
//
// One read pass computes both the plain and the inverted popcount of every
// chunk, so the complement decision, the chunk->container map and all
// metadata are produced on the device and the call needs a single host sync.
#include <algorithm>

#include "internal.hpp"

namespace crimpl {

constexpr int BS_NT = 256;

// What the call reads back.
struct BsTotals {
    uint32_t n_containers;
    uint32_t negated;
    uint32_t max_key;
    unsigned long long total;  // popcount of the input
};

// A workgroup's chunks together: their popcount, and how many are kept
// (non-empty) as they are and inverted.
struct alignas(16) BsPart {
    uint32_t total;  // at most BS_PER chunks of 65536
    uint32_t kept, kept_inv;
};

struct BsGeom {
    uint32_t n_words;
    uint32_t n_chunks;
    uint32_t per;        // consecutive chunks of a workgroup, at most BS_PER
    uint32_t tail_idx;   // word masked after inversion, or 0xFFFFFFFF
    uint32_t tail_mask;
    uint32_t universe;
};

__device__ __forceinline__ uint32_t load_word(const uint32_t* w, uint32_t i, uint32_t n) { return i < n ? w[i] : 0u; }

// Both kernels give workgroup b the chunks [b per, b per + per).  65536 chunks on
// the 8 workgroups a CU of a 256-CU device are 32 each.
constexpr uint32_t BS_PER = 64;      // chunk flags of a workgroup fit one ballot
constexpr uint32_t BS_GROUPS = 4096;  // workgroups at most (bs_compact reads every one's counts)

__device__ __forceinline__ bool bs_whole(const uint32_t* words, const BsGeom& g, uint32_t base)
{
    return base + 2048u <= g.n_words && (reinterpret_cast<uintptr_t>(words + base) & 15u) == 0;
}

// Per chunk: popcount of the words and of their inversion (tail word masked,
// words past n_words are zero in both); a wave takes a chunk.
__global__ __launch_bounds__(BS_NT) void bs_count(const uint32_t* __restrict__ words, BsGeom g, uint32_t* pc,
                                                  uint32_t* pci, BsPart* part)
{
    __shared__ uint32_t s_total, s_kept, s_inv;
    if (threadIdx.x == 0) s_total = 0, s_kept = 0, s_inv = 0;
    __syncthreads();
    const uint32_t lane = __lane_id();
    const uint32_t c0 = blockIdx.x * g.per, c1 = min(g.n_chunks, c0 + g.per);
    for (uint32_t c = c0 + (threadIdx.x >> 6); c < c1; c += BS_NT / 64) {
        const uint32_t base = c * 2048u;
        uint32_t a = 0, b = 0;
        if (bs_whole(words, g, base)) {
            // Ordinary loads: the bitset (U/8 bytes, 128 MiB at 2^30) stays in
            // the Infinity Cache for bs_compact, which reads it again.
            const uint4* s4 = reinterpret_cast<const uint4*>(words + base);
            uint4 v[8];
#pragma unroll
            for (int h = 0; h < 8; ++h) v[h] = s4[lane + 64 * h];
#pragma unroll
            for (int h = 0; h < 8; ++h) a += __popc(v[h].x) + __popc(v[h].y) + __popc(v[h].z) + __popc(v[h].w);
            b = 8u * 128u - a;
            if (g.tail_idx - base < 2048u) {  // (unsigned) the tail word's bits past the universe are no ids of the inversion
                const uint32_t w = g.tail_idx - base;
                if ((w / 4u) % 64u == lane) b -= 32u - __popc(g.tail_mask) - __popc(words[g.tail_idx] & ~g.tail_mask);
            }
        } else {
            for (uint32_t k = lane; k < 2048u; k += 64) {
                const uint32_t i = base + k;
                if (i < g.n_words) {
                    const uint32_t w = words[i];
                    a += __popc(w);
                    b += (i == g.tail_idx) ? __popc(~w & g.tail_mask) : 32u - __popc(w);
                }
            }
        }
        a = wave_sum(a);
        b = wave_sum(b);
        if (lane == 0) {
            pc[c] = a;
            pci[c] = b;
            atomicAdd(&s_total, a);
            if (a) atomicAdd(&s_kept, 1u);
            if (b) atomicAdd(&s_inv, 1u);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        BsPart r;
        r.total = s_total, r.kept = s_kept, r.kept_inv = s_inv;
        part[blockIdx.x] = r;
    }
}

// Plans and copies.  Every workgroup sums all workgroups' counts itself (16 bytes
// each, at most 64 KiB from the L2): the whole popcount decides the negation
// (total > U/2, strict, src/upload_ids.cu:837), and the kept chunks before its own
// give their ranks, so nothing waits for another kernel or workgroup.  It writes
// its chunks' keys, types, offsets, cards and key_index and copies (or inverts)
// the kept ones; the workgroup of the last kept chunk writes the totals into
// the caller's pinned host slot.  A separate planning kernel of one workgroup per
// 1024 chunks took 13 us and a launch: at 10^9 bits the three kernels took 73 us
// (the call 82.6), these two 66 (77.9); at 2^30 78 (87.8) and 66 (78.8).
__global__ __launch_bounds__(BS_NT) void bs_compact(const uint32_t* __restrict__ words, BsGeom g, const uint32_t* pc,
                                                    const uint32_t* pci, const BsPart* part, uint16_t* keys,
                                                    uint8_t* types, uint32_t* offsets, uint16_t* cards,
                                                    uint16_t* key_index, uint64_t* __restrict__ pool, BsTotals* host)
{
    constexpr int NW = BS_NT / 64;
    __shared__ unsigned long long s_sum[NW];
    __shared__ uint32_t s_cnt[4][NW];  // kept and kept inverted, before this workgroup and in all
    __shared__ uint32_t s_rank[BS_PER];
    const uint32_t t = threadIdx.x, lane = __lane_id(), wave = t >> 6;
    const uint32_t c0 = blockIdx.x * g.per, c1 = min(g.n_chunks, c0 + g.per);
    // The first chunk's words, on their way while the counts are summed.
    const bool first_whole = bs_whole(words, g, c0 * 2048u);
    uint4 first[2] = {};
    if (first_whole) {
        const uint4* s4 = reinterpret_cast<const uint4*>(words + c0 * 2048u);
#pragma unroll
        for (int h = 0; h < 2; ++h) first[h] = ld_stream(s4 + t + h * BS_NT);
    }
    const uint32_t own_p = t < c1 - c0 ? pc[c0 + t] : 0u, own_i = t < c1 - c0 ? pci[c0 + t] : 0u;
    unsigned long long sum = 0;
    uint32_t n[4] = {0, 0, 0, 0};
    for (uint32_t i0 = t; i0 < gridDim.x; i0 += 8 * BS_NT) {
        BsPart r[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = i0 + k * BS_NT < gridDim.x ? part[i0 + k * BS_NT] : BsPart{};
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool before = i0 + k * BS_NT < blockIdx.x;
            sum += r[k].total;
            n[0] += before ? r[k].kept : 0u;
            n[1] += before ? r[k].kept_inv : 0u;
            n[2] += r[k].kept;
            n[3] += r[k].kept_inv;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
#pragma unroll
    for (int k = 0; k < 4; ++k) n[k] = wave_sum(n[k]);
    if (lane == 0) {
        s_sum[wave] = sum;
#pragma unroll
        for (int k = 0; k < 4; ++k) s_cnt[k][wave] = n[k];
    }
    __syncthreads();
    unsigned long long total = 0;
    uint32_t base_p = 0, base_i = 0, all_p = 0, all_i = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        total += s_sum[w];
        base_p += s_cnt[0][w], base_i += s_cnt[1][w], all_p += s_cnt[2][w], all_i += s_cnt[3][w];
    }
    const bool negate = total > static_cast<unsigned long long>(g.universe / 2u);  // :837
    const uint32_t all = negate ? all_i : all_p;
    if (wave == 0) {  // a lane per chunk
        const uint32_t v = negate ? own_i : own_p, c = c0 + lane;
        const unsigned long long m = __ballot(v != 0u);
        const uint32_t rank = (negate ? base_i : base_p) + static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
        if (lane < BS_PER) s_rank[lane] = v != 0u ? rank : 0xFFFFFFFFu;
        if (c < c1) key_index[c] = v != 0u ? static_cast<uint16_t>(rank) : uint16_t(0xFFFFu);
        if (v != 0u) {
            keys[rank] = static_cast<uint16_t>(c);
            types[rank] = CR_BITMAP;
            offsets[rank] = rank * 8192u;
            cards[rank] = static_cast<uint16_t>(v > 65535u ? 0u : v);
        }
        if ((v != 0u && rank == all - 1u) || (all == 0u && blockIdx.x == 0 && lane == 0)) {
            volatile BsTotals* h = host;
            h->n_containers = all;
            h->negated = negate ? 1u : 0u;
            h->max_key = all ? c : 0u;
            h->total = total;
        }
    }
    __syncthreads();
    for (uint32_t c = c0; c < c1; ++c) {
        const uint32_t r = s_rank[c - c0];
        if (r == 0xFFFFFFFFu) continue;
        uint32_t* dst = reinterpret_cast<uint32_t*>(pool) + static_cast<uint64_t>(r) * 2048u;
        const uint32_t base = c * 2048u;
        if (bs_whole(words, g, base)) {
            const uint4* s4 = reinterpret_cast<const uint4*>(words + base);
            uint4* d4 = reinterpret_cast<uint4*>(dst);
            uint4 v[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) v[h] = c == c0 ? first[h] : ld_stream(s4 + t + h * BS_NT);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (negate) {
                    const uint32_t i0 = base + 4u * (t + h * BS_NT);
                    v[h] = make_uint4(~v[h].x, ~v[h].y, ~v[h].z, ~v[h].w);
                    if (i0 == g.tail_idx) v[h].x &= g.tail_mask;
                    if (i0 + 1 == g.tail_idx) v[h].y &= g.tail_mask;
                    if (i0 + 2 == g.tail_idx) v[h].z &= g.tail_mask;
                    if (i0 + 3 == g.tail_idx) v[h].w &= g.tail_mask;
                }
                st_stream(d4 + t + h * BS_NT, v[h]);
            }
        } else {
            for (uint32_t k = t; k < 2048u; k += BS_NT) {
                const uint32_t i = base + k;
                uint32_t w = 0;
                if (i < g.n_words) {
                    w = words[i];
                    if (negate) {
                        w = ~w;
                        if (i == g.tail_idx) w &= g.tail_mask;
                    }
                }
                dst[k] = w;
            }
        }
    }
}

int upload_from_device_bitset_impl(const uint32_t* d_words, uint32_t n_words, uint32_t universe, hipStream_t s,
                                   cr_gpu_roaring* out)
{
    reset(out);
    out->universe_size = universe;
    if (n_words == 0) return CR_OK;  // src/upload_ids.cu:811-815
    BsGeom g{};
    g.n_words = n_words;
    g.n_chunks = static_cast<uint32_t>((static_cast<uint64_t>(n_words) + 2047u) / 2048u);
    if (g.n_chunks > 65536u) {
        set_error("upload_from_device_bitset: %u words exceed the 2^32-id key space", n_words);
        return CR_ERR_UNSUPPORTED;
    }
    g.universe = universe;
    const uint32_t tail_bits = universe % 32u;  // :851-858
    g.tail_idx = (tail_bits > 0 && universe / 32u < n_words) ? universe / 32u : 0xFFFFFFFFu;
    g.tail_mask = tail_bits ? ((1u << tail_bits) - 1u) : ~0u;

    const uint32_t want = std::max(1u, std::min<uint32_t>(BS_GROUPS, num_cus() * 8u));  // workgroups
    g.per = (g.n_chunks + want - 1) / want;
    if (g.per > BS_PER) g.per = BS_PER;  // (65536 chunks in BS_PER each are 1024 workgroups)
    const unsigned grid = (g.n_chunks + g.per - 1) / g.per;

    Carver c;
    const size_t o_pc = c.add(4ull * g.n_chunks);
    const size_t o_pci = c.add(4ull * g.n_chunks);
    const size_t o_part = c.add(sizeof(BsPart) * grid);
    Scratch sc;
    CR_RET(sc.alloc(c.total, s));
    uint32_t* pc = sc.at<uint32_t>(o_pc);
    uint32_t* pci = sc.at<uint32_t>(o_pci);
    BsPart* part = sc.at<BsPart>(o_part);

    const OutLayout L = plan_out(g.n_chunks, g.n_chunks, static_cast<uint64_t>(g.n_chunks) * 1024u, 0, 0);
    CR_RET(alloc_out(out, L, g.n_chunks, g.n_chunks, static_cast<uint64_t>(g.n_chunks) * 1024u, 0, 0, s));

    {
        CR_TIMED("bs_count", s);
        bs_count<<<grid, BS_NT, 0, s>>>(d_words, g, pc, pci, part);
    }
    CR_LAUNCH_CHECK();
    HostSlotGuard hs;
    CR_RET(hs.acquire());
    {
        CR_TIMED("bs_compact", s);
        bs_compact<<<grid, BS_NT, 0, s>>>(d_words, g, pc, pci, part, out->keys, out->types, out->offsets,
                                          out->cardinalities, out->key_index, out->bitmap_data, hs.dev<BsTotals>());
    }
    CR_LAUNCH_CHECK();
    CR_RET(sync_stream(s));
    BsTotals h{};
    {
        const volatile BsTotals* hp = hs.host<BsTotals>();
        h.n_containers = hp->n_containers;
        h.negated = hp->negated;
        h.max_key = hp->max_key;
        h.total = hp->total;
    }
    out->negated = h.negated != 0;
    out->total_cardinality = h.total;  // logical count either way (:740)
    out->n_containers = h.n_containers;
    out->n_bitmap_containers = h.n_containers;
    if (h.n_containers == 0) {  // no key_index on an empty result (:747-750)
        free_async(out, s);
        out->universe_size = universe;
        out->negated = h.negated != 0;
        out->total_cardinality = h.total;
        return CR_OK;
    }
    out->max_key = h.max_key;
    return CR_OK;
}

}  // namespace crimpl

using namespace crimpl;

extern "C" int cr_upload_from_device_bitset(const uint32_t* d_words, uint32_t n_words, uint32_t universe_size,
                                            cr_stream_t stream, cr_gpu_roaring* out)
{
    if (!out || (n_words && !d_words)) {
        set_error("cr_upload_from_device_bitset: invalid argument");
        return CR_ERR_INVALID;
    }
    reset(out);
    return produced(upload_from_device_bitset_impl(d_words, n_words, universe_size, as_stream(stream), out), out,
                    as_stream(stream));
}

extern "C" int cr_upload_from_bitset(const uint32_t* host_words, uint32_t n_words, uint32_t universe_size,
                                     cr_stream_t stream, cr_gpu_roaring* out)
{
    if (!out || (n_words && !host_words)) {
        set_error("cr_upload_from_bitset: invalid argument");
        return CR_ERR_INVALID;
    }
    hipStream_t s = as_stream(stream);
    reset(out);
    if (n_words == 0) return produced(upload_from_device_bitset_impl(nullptr, 0, universe_size, s, out), out, s);
    Scratch sc;
    CR_RET(sc.alloc(static_cast<size_t>(n_words) * 4u, s));
    CR_RET(h2d_pageable(sc.ptr, host_words, static_cast<size_t>(n_words) * 4u, s));
    return produced(upload_from_device_bitset_impl(sc.at<uint32_t>(0), n_words, universe_size, s, out), out, s);
}
