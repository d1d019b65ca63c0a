// hb_union.h -- the per-node HyperBall union step shared by the single-graph
// kernels (hb_kernels.hip) and the batched kernels (hb_batch.hip).
//
// For node u (hyper_ball.rs:803-831): a = c_{t-1}(u) | c_{t-1}(v) for every
// neighbour v; est(a) against the cached est(c_{t-1}(u)); f64 accumulation when
// the estimate increased; c_t(u) = a into the output buffer; changed-bit when any
// register changed.  A team of T lanes runs one node: G = 2^P/16 lanes hold one
// sketch copy (16 registers each), S = T/G copies split the neighbour list.
#pragma once

#include "hb_device.h"

namespace hb {

// What an iteration reads of the neighbours.  Each kind is a kernel of its own: together
// in one, they cost every one of them registers (k_union<7, 8> spills 10 VGPRs at eight
// wavefronts per SIMD with all three, none with the first iteration's apart) and LDS.
enum class Gather {
    kAll,      // every neighbour's registers
    kChanged,  // those of the neighbours in HbView::gather_bits
    kFirst,    // iteration 1: sketches hold only their own insertion, so ids are hashed
};

// one graph's state as seen by one iteration
struct HbView {
    const uint32_t *off, *nbr;
    const uint32_t *orig;      // hashed id of each arc's head (iteration 1)
    const uint32_t *node_id;   // hashed id of each node (null: its index)
    const uint8_t *in;
    uint32_t *scr;          // LDS; Gather::kFirst with P <= 10: 16 u32 per lane of the block
    uint8_t *out;
    float *est;
    double *dist, *inv;
    const uint32_t *bitsR;  // registers changed at t-1
    const uint32_t *gather_bits;  // bitsR when only changed neighbours need gathering, else null
    uint32_t *bitsW;        // registers changed at t
    double t, inv_t;
    bool use_frontier;
    // saturation (null: not used in this iteration): the nodes whose sketch is the upper
    // bound of all sketches at t-1 and at t, and the bound itself (LDS, G uint4)
    const uint32_t *satR = nullptr;
    uint32_t *satW = nullptr;
    const uint4 *bound = nullptr;
    bool sat_scan = false;  // look for a saturated neighbour before the gather
    bool sym = false;
};

// One lane's counts over its share of a launch.  32 bits suffice (a lane's sums are at
// most the graph's node or arc count, both below 2^32 in the u32 CSR) and keep five
// registers free in the union kernels; the block and batch sums widen them to 64 bits.
struct HbCounts {
    uint32_t inc = 0, arcs = 0, nodes = 0, chg = 0;
    uint32_t gathered = 0;  // neighbour register blocks read
    uint32_t sat = 0;       // degrees of the nodes that became saturated
};

__device__ __forceinline__ bool bit_test(const uint32_t *bits, uint32_t v)
{
    return (bits[v >> 5] >> (v & 31u)) & 1u;
}

// f64 accumulation without contraction (hyper_ball.rs:819-828); dist0 / inv0 are the
// node's accumulators as loaded by the caller
__device__ __forceinline__ bool accumulate(const HbView &v, uint32_t u, float prev, float curr, double dist0,
                                           double inv0)
{
    const float d32 = __fsub_rn(curr, prev);
    const double diff = (double)d32;
    if (diff > 0.0) {
        v.dist[u] = __dadd_rn(dist0, __dmul_rn(v.t, diff));
        v.inv[u] = __dadd_rn(inv0, __dmul_rn(v.inv_t, diff));
        return true;
    }
    return false;
}
__device__ __forceinline__ bool accumulate(const HbView &v, uint32_t u, float prev, float curr)
{
    const float d32 = __fsub_rn(curr, prev);
    if (!((double)d32 > 0.0)) return false;  // the accumulators are read only when needed
    return accumulate(v, u, prev, curr, v.dist[u], v.inv[u]);
}

// 16 bytes of a new register row.  A row is next read an iteration later, after all the others:
// written as streaming data it leaves L2 to the rows that are gathered (k_union_rows on the k-mer
// graph 294 -> 282 us a launch; iterations of R-MAT-20 at p = 8 1.4% shorter, of R-MAT-24
// 0.6%; graphs whose rows all stay in L2: no difference)
typedef uint32_t hb_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_row(uint4 *p, uint4 r)
{
    __builtin_nontemporal_store(hb_u32x4{r.x, r.y, r.z, r.w}, (hb_u32x4 *)p);
}

// (index << 6) | rank of the insertion of node id v at precision P (P <= 10)
template <int P>
__device__ __forceinline__ uint32_t hb_insertion(uint32_t v)
{
    uint32_t idx, rank;
    hb_index_rank(v, P, &idx, &rank);
    return (idx << 6) | rank;
}

// This lane's 16 registers of c_0(v) for copy lane cl, from w = (index << 6) | rank.
__device__ __forceinline__ uint4 hb_own_from_word(uint32_t w, uint32_t cl)
{
    const uint32_t idx = w >> 6, rank = w & 63u;
    uint4 r = make_uint4(0, 0, 0, 0);
    if ((idx >> 4) == cl) {
        const uint32_t v = rank << (8u * (idx & 3u)), q = (idx >> 2) & 3u;
        r.x = q == 0 ? v : 0u;
        r.y = q == 1 ? v : 0u;
        r.z = q == 2 ? v : 0u;
        r.w = q == 3 ? v : 0u;
    }
    return r;
}

// register idx of the copy := max(register, rank) when it falls in lane cl's 16
__device__ __forceinline__ void hb_put_max(uint4 &a, uint32_t w, uint32_t cl)
{
    const uint32_t idx = w >> 6;
    if ((idx >> 4) != cl) return;
    const uint32_t sh = 8u * (idx & 3u), q = (idx >> 2) & 3u;
    const uint32_t m = 0xffu << sh, r = (w & 63u) << sh;
    uint32_t x = q == 0 ? a.x : q == 1 ? a.y : q == 2 ? a.z : a.w;
    if ((x & m) < r) x = (x & ~m) | r;
    if (q == 0) a.x = x;
    else if (q == 1) a.y = x;
    else if (q == 2) a.z = x;
    else a.w = x;
}

// Union of the sketches of nb[slot], nb[slot + S], ... (j < len) into `start`,
// for the 16 registers of copy lane cl (the copy is G = 2^P/16 consecutive lanes).
// kChanged: only the neighbours in `changed` (the nodes whose registers changed at t-1) are
// gathered: an unchanged neighbour v has c_{t-1}(v) = c_{t-2}(v), which c_{t-1}(u)
// already contains (v is u's neighbour), so leaving it out changes nothing.
// kFirst: in iteration 1 every neighbour's sketch is still its own insertion, so
// instead of gathering its 2^P-byte register block the copy's lanes hash the
// neighbour ids, one each, and raise register idx to the rank with an LDS atomic max
// on a u32 per register (`scr`: 16 u32 per lane, the copy's registers contiguous
// from the copy's first lane); no random global memory access at all.
template <int P, uint32_t S, Gather kGather>
__device__ __forceinline__ uint4 hb_gather_union(const uint8_t *__restrict__ in, uint32_t *scr,
                                                 const uint32_t *__restrict__ changed,
                                                 const uint32_t *__restrict__ nb,
                                                 const uint32_t *__restrict__ nbh, uint32_t len, uint32_t slot,
                                                 uint32_t cl, uint4 start, uint32_t &gathered)
{
    constexpr uint32_t G = (1u << P) / 16;
    uint32_t j = slot;
    if constexpr (kGather == Gather::kFirst) {
        uint32_t *mine = scr + threadIdx.x * 16u;              // this lane's 16 registers
        uint32_t *copy = scr + (threadIdx.x - cl) * 16u;       // register idx of the copy at copy[idx]
        const uint32_t sw[4] = {start.x, start.y, start.z, start.w};
#pragma unroll
        for (int k = 0; k < 16; ++k) mine[k] = (sw[k >> 2] >> (8 * (k & 3))) & 0xffu;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t q = slot + cl * S; q < len; q += G * S) {
            const uint32_t w = hb_insertion<P>(nbh[q]);
            atomicMax(copy + (w >> 6), w & 63u);
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            r[k] = mine[4 * k] | (mine[4 * k + 1] << 8) | (mine[4 * k + 2] << 16) | (mine[4 * k + 3] << 24);
        return make_uint4(r[0], r[1], r[2], r[3]);
    }
    HbAcc pa = hb_acc(start);
    if constexpr (kGather == Gather::kChanged) {
        const uint4 z = make_uint4(0, 0, 0, 0);  // registers are >= 0: max with 0 is a no-op
        for (; j + 3 * S < len; j += 4 * S) {
            const uint32_t v0 = nb[j], v1 = nb[j + S], v2 = nb[j + 2 * S], v3 = nb[j + 3 * S];
            const bool c0 = bit_test(changed, v0), c1 = bit_test(changed, v1);
            const bool c2 = bit_test(changed, v2), c3 = bit_test(changed, v3);
            gathered += (uint32_t)c0 + (uint32_t)c1 + (uint32_t)c2 + (uint32_t)c3;
            const uint4 x0 = c0 ? *(const uint4 *)(in + ((uint64_t)v0 << P) + cl * 16) : z;
            const uint4 x1 = c1 ? *(const uint4 *)(in + ((uint64_t)v1 << P) + cl * 16) : z;
            const uint4 x2 = c2 ? *(const uint4 *)(in + ((uint64_t)v2 << P) + cl * 16) : z;
            const uint4 x3 = c3 ? *(const uint4 *)(in + ((uint64_t)v3 << P) + cl * 16) : z;
            hb_acc_max(pa, x0);
            hb_acc_max(pa, x1);
            hb_acc_max(pa, x2);
            hb_acc_max(pa, x3);
        }
        for (; j < len; j += S) {
            const uint32_t v = nb[j];
            if (bit_test(changed, v)) {
                hb_acc_max(pa, *(const uint4 *)(in + ((uint64_t)v << P) + cl * 16));
                ++gathered;
            }
        }
        return hb_acc_get(pa);
    } else {
        (void)changed;
    }
    gathered += len > slot ? (len - slot + S - 1) / S : 0;
    for (; j + 3 * S < len; j += 4 * S) {
        const uint32_t v0 = nb[j], v1 = nb[j + S], v2 = nb[j + 2 * S], v3 = nb[j + 3 * S];
        const uint4 x0 = *(const uint4 *)(in + ((uint64_t)v0 << P) + cl * 16);
        const uint4 x1 = *(const uint4 *)(in + ((uint64_t)v1 << P) + cl * 16);
        const uint4 x2 = *(const uint4 *)(in + ((uint64_t)v2 << P) + cl * 16);
        const uint4 x3 = *(const uint4 *)(in + ((uint64_t)v3 << P) + cl * 16);
        hb_acc_max(pa, x0);
        hb_acc_max(pa, x1);
        hb_acc_max(pa, x2);
        hb_acc_max(pa, x3);
    }
    for (; j < len; j += S) hb_acc_max(pa, *(const uint4 *)(in + ((uint64_t)nb[j] << P) + cl * 16));
    return hb_acc_get(pa);
}

// Whether one of the first neighbours of a list is saturated, asked by a team of T lanes
// (all of them return it).  The degree layout lists the high-degree nodes, which saturate
// first, at the front, so a node with a saturated neighbour nearly always shows it within
// the first 2 T ids; missing one only costs the gather.
template <int T>
__device__ __forceinline__ bool sat_neighbour(const uint32_t *__restrict__ sat, const uint32_t *__restrict__ nb,
                                              uint32_t len, uint32_t tl, uint32_t &scanned)
{
    for (uint32_t k = 0; k < 2 && k * T < len; ++k) {
        const uint32_t j = k * T + tl;
        scanned = min(len, (k + 1) * T);
        if (hb_copy_or<T>(j < len ? (uint32_t)bit_test(sat, nb[j]) : 0u)) return true;
    }
    return false;
}

// Whether a node whose sketch is the bound is to be marked saturated.  Two nodes that are
// each other's only neighbour are left out of the bound (k_init), so neither is marked.
__device__ __forceinline__ bool sat_allowed(const HbView &v, const uint32_t *nb, uint32_t deg)
{
    return !(v.sym && deg == 1 && v.off[nb[0] + 1] - v.off[nb[0]] == 1);
}

__device__ __forceinline__ void bit_set(uint32_t *bits, uint32_t u) { atomicOr(bits + (u >> 5), 1u << (u & 31u)); }

// The nodes u0 + team, team = 0 .. 64 / T - 1 of the wavefront, whose teams have `set`
// (the same on every lane of a team), ORed into a bitmap with one atomic per word.  One per
// node had the 8 or 16 nodes of a wavefront queue on one word: R-MAT-24 (p = 7) 23.6 ms per
// run against 21.8, ER (n = 65,536, p = 6) 0.37 against 0.30.
template <int T>
__device__ __forceinline__ void bits_set(uint32_t *bits, uint32_t u0, bool set)
{
    uint64_t m = __ballot(set);
    if (m == 0) return;
    if constexpr (T == 2) {  // every T-th bit, packed
        m &= 0x5555555555555555ull;
        m = (m | m >> 1) & 0x3333333333333333ull;
        m = (m | m >> 2) & 0x0f0f0f0f0f0f0f0full;
        m = (m | m >> 4) & 0x00ff00ff00ff00ffull;
        m = (m | m >> 8) & 0x0000ffff0000ffffull;
        m = (m | m >> 16) & 0xffffffffull;
    } else if constexpr (T == 4) {
        m &= 0x1111111111111111ull;
        m = (m | m >> 3) & 0x0303030303030303ull;
        m = (m | m >> 6) & 0x000f000f000f000full;
        m = (m | m >> 12) & 0x000000ff000000ffull;
        m = (m | m >> 24) & 0xffffull;
    } else if constexpr (T == 8) {
        m = ((m & 0x0101010101010101ull) * 0x0102040810204080ull) >> 56;
    } else if constexpr (T >= 16) {
        uint64_t x = 0;
#pragma unroll
        for (int k = 0; k < HB_WAVE / T; ++k) x |= ((m >> (k * T)) & 1ull) << k;
        m = x;
    }
    const uint32_t sh = u0 & 31u, lane = threadIdx.x & (HB_WAVE - 1);
    const uint64_t lo = m << sh, hi = T == 1 && sh ? m >> (64 - sh) : 0ull;
    const uint32_t w = lane == 0 ? (uint32_t)lo : lane == 1 ? (uint32_t)(lo >> 32) : (uint32_t)hi;
    if (lane < 3 && w) atomicOr(bits + (u0 >> 5) + lane, w);
}

// Returns, on every lane of the team, kChangedBit when a register rose and kSaturatedBit when
// the node is to be marked saturated; the caller sets the bitmaps.
constexpr uint32_t kChangedBit = 1, kSaturatedBit = 2;

template <int P, int T, Gather kGather>
__device__ __forceinline__ uint32_t union_node(const HbView &v, const HbTables &tb, uint32_t u, uint32_t tl,
                                               HbCounts &c)
{
    constexpr uint32_t M = 1u << P, G = M / 16, S = T / G;
    static_assert(T >= (int)G && T <= HB_WAVE, "team width");
    (void)M;
    const uint32_t cl = tl % G, slot = tl / G;
    const uint32_t e0 = v.off[u], deg = v.off[u + 1] - e0;
    const uint32_t *__restrict__ nb = v.nbr + e0;
    const uint32_t *__restrict__ nbh = v.orig + e0;
    bool sat = false;  // a neighbour is saturated, so this node becomes so
    uint32_t scanned = deg;
    if (kGather != Gather::kFirst && v.satR) {
        if (bit_test(v.satR, u)) {  // nothing can change; keep both buffers complete
            if (slot == 0 && bit_test(v.bitsR, u)) *(uint4 *)(v.out + ((uint64_t)u << P) + cl * 16) = v.bound[cl];
            return 0;
        }
        if (v.sat_scan) {
            uint32_t k = 0;
            sat = sat_neighbour<T>(v.satR, nb, deg, tl, k);
            if (sat) scanned = k;
        }
    }
    if (kGather == Gather::kChanged && v.use_frontier && !sat) {
        uint32_t any = 0;
        for (uint32_t j = tl; j < deg; j += T) any |= bit_test(v.bitsR, nb[j]);
        if (hb_copy_or<T>(any) == 0) {
            // no neighbour changed: c_t(u) = c_{t-1}(u); keep both buffers complete
            if (slot == 0 && bit_test(v.bitsR, u))
                *(uint4 *)(v.out + ((uint64_t)u << P) + cl * 16) =
                    *(const uint4 *)(v.in + ((uint64_t)u << P) + cl * 16);
            return 0;
        }
    }
    uint4 acc;
    uint32_t diffw;  // bit 0: a register rose; bit 1: a register is below the bound
    if (sat) {
        acc = v.bound[cl];
        diffw = 1u;  // this one is not marked, so it is below the bound and rises
    } else {
        uint4 own;
        if constexpr (kGather == Gather::kFirst)
            own = hb_own_from_word(hb_insertion<P>(v.node_id ? v.node_id[u] : u), cl);
        else
            own = *(const uint4 *)(v.in + ((uint64_t)u << P) + cl * 16);
        uint32_t gathered = 0;  // by this lane's copy
        acc = hb_gather_union<P, S, kGather>(v.in, v.scr, v.gather_bits, nb, nbh, deg, slot, cl, own, gathered);
        if (cl == 0) c.gathered += gathered;
#pragma unroll
        for (uint32_t s = G; s < T; s <<= 1) acc = hb_bmax4(acc, hb_shfl_xor4<T>(acc, s));
        diffw = (acc.x != own.x) | (acc.y != own.y) | (acc.z != own.z) | (acc.w != own.w);
        if (kGather != Gather::kFirst && v.satR) {
            const uint4 f = v.bound[cl];
            diffw |= ((acc.x != f.x) | (acc.y != f.y) | (acc.z != f.z) | (acc.w != f.w)) << 1;
        }
        diffw = hb_copy_or<G>(diffw);
    }
    uint32_t r = diffw & 1u ? kChangedBit : 0u;
    if (kGather != Gather::kFirst && v.satR && !(diffw & 2u) && sat_allowed(v, nb, deg)) r |= kSaturatedBit;
    const float curr = hb_estimate_copy<G>(tb, acc);
    if (slot == 0) store_row((uint4 *)(v.out + ((uint64_t)u << P) + cl * 16), acc);
    if (tl == 0) {
        const float prev = v.est[u];
        if (accumulate(v, u, prev, curr)) c.inc += 1;
        v.est[u] = curr;
        if (r & kChangedBit) c.chg += 1;
        if (r & kSaturatedBit) c.sat += deg;
        c.arcs += scanned;
        c.nodes += 1;
    }
    return r;
}

// union_node of the consecutive nodes u0 + team (team < count) by the wavefront's teams
template <int P, int T, Gather kGather>
__device__ __forceinline__ void union_wave(const HbView &v, const HbTables &tb, uint32_t u0, uint32_t count,
                                           HbCounts &c)
{
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    const uint32_t r = lane / T < count ? union_node<P, T, kGather>(v, tb, u0 + lane / T, lane % T, c) : 0u;
    bits_set<T>(v.bitsW, u0, (r & kChangedBit) != 0);
    if (kGather != Gather::kFirst && v.satR) bits_set<T>(v.satW, u0, (r & kSaturatedBit) != 0);
}

// union_node for a dense iteration (every neighbour gathered, no frontier check) with one
// sketch copy per team (T = G), where the wavefront's 64 / G teams hold the consecutive
// nodes lo .. hi - 1 (a bin that is an id range).  Each team puts its own row into the
// wavefront's LDS window `win` (64 uint4, copy lane cl of node w at (w - lo) G + cl), and a
// neighbour inside [lo, hi) is read from there instead of memory: in a numbering that
// keeps chains together (the chain layout) most neighbours are in the window, and the
// union is bound by the rate of memory requests, not by bytes.  Same registers,
// estimates and accumulators as union_node.  (At p = 5 and 6 the single-graph engine runs
// such iterations with one node per lane instead: k_union_rows.)
template <int P, int T>
__device__ __forceinline__ void union_node_window(const HbView &v, const HbTables &tb, uint32_t u, uint32_t tl,
                                                  HbCounts &c, uint32_t lo, uint32_t hi, uint4 *win)
{
    constexpr uint32_t G = (1u << P) / 16;
    static_assert(T == (int)G, "one copy per team");
    const uint32_t cl = tl;
    const uint32_t e0 = v.off[u], deg = v.off[u + 1] - e0;
    const uint32_t *__restrict__ nb = v.nbr + e0;
    const uint8_t *__restrict__ in = v.in;
    // the node's estimate is loaded beside its own row, its accumulators right after the
    // gathers: each then arrives while the union and the estimate are computed instead of
    // costing a memory round trip of its own after them (≈ 1% on the k-mer graph)
    const float prev = tl == 0 ? v.est[u] : 0.0f;
    const uint4 own = *(const uint4 *)(in + ((uint64_t)u << P) + cl * 16);
    win[(u - lo) * G + cl] = own;
    // LDS operations of one wavefront complete in order; the barrier and fence keep the
    // compiler from moving the window reads above the write
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t span = hi - lo;
    HbAcc pa = hb_acc(own);
    uint32_t j = 0;
    for (; j + 1 < deg; j += 2) {
        const uint32_t w0 = nb[j], w1 = nb[j + 1];
        const uint4 x0 = w0 - lo < span ? win[(w0 - lo) * G + cl] : *(const uint4 *)(in + ((uint64_t)w0 << P) + cl * 16);
        const uint4 x1 = w1 - lo < span ? win[(w1 - lo) * G + cl] : *(const uint4 *)(in + ((uint64_t)w1 << P) + cl * 16);
        hb_acc_max(pa, x0);
        hb_acc_max(pa, x1);
    }
    if (j < deg) {
        const uint32_t w0 = nb[j];
        hb_acc_max(pa, w0 - lo < span ? win[(w0 - lo) * G + cl] : *(const uint4 *)(in + ((uint64_t)w0 << P) + cl * 16));
    }
    const uint4 acc = hb_acc_get(pa);
    double dist0 = 0.0, inv0 = 0.0;
    if (tl == 0) {
        dist0 = v.dist[u];
        inv0 = v.inv[u];
    }
    if (cl == 0) c.gathered += deg;
    // every team has read the window before the next trip overwrites it
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    const uint32_t diffw = (acc.x != own.x) | (acc.y != own.y) | (acc.z != own.z) | (acc.w != own.w);
    const bool changed = hb_copy_or<G>(diffw) != 0;
    const float curr = hb_estimate_copy<G>(tb, acc);
    *(uint4 *)(v.out + ((uint64_t)u << P) + cl * 16) = acc;
    if (tl == 0) {
        if (accumulate(v, u, prev, curr, dist0, inv0)) c.inc += 1;
        v.est[u] = curr;
        if (changed) {
            atomicOr(v.bitsW + (u >> 5), 1u << (u & 31u));
            c.chg += 1;
        }
        c.arcs += deg;
        c.nodes += 1;
    }
}

}  // namespace hb
