// hb_kernels.hip -- HyperBall iteration kernels for gfx950 (no MFMA: the union
// is a bytewise max, HBM-bound).
//
// One iteration t (hyper_ball.rs:754-874, restated per node u):
//     a = c_{t-1}(u); for v in N(u): a |= c_{t-1}(v)       (register-wise max)
//     diff = f64(est(a) - est(c_{t-1}(u)))  (f32 subtraction)
//     if diff > 0 { dist[u] += t*diff; inv[u] += (1/t)*diff; increases++ }
//     c_t(u) = a
// Launch sequence per iteration, all reading the device-resident HbIterState so
// that one captured hipGraph serves every iteration:
//     k_begin (clear next changed-bitmap)  ->  k_union<P,T,kFirst> per degree bin
//     (k_union_rows<P> for the dense iterations of a chain-layout id range at p = 5, 6)
//     ->  k_chunk<P,kFirst> (hub neighbour chunks) -> k_merge<P> (hubs) -> [k_nf] -> k_finalize
// Frontier: if no neighbour of u changed at t-1 then c_t(u) = c_{t-1}(u) (union
// of unchanged sets), so u is skipped; when u itself changed at t-1 its row is
// copied into the output buffer so both buffers stay complete.  Results are
// identical to recomputing every node.
// Saturation: no sketch exceeds the register-wise maximum B of all insertions (k_init; on
// a symmetric graph without those that reach no other node).  A node whose sketch is B is
// done for good, and a node with such a neighbour becomes B whatever the others hold, so
// neither gathers anything.  Graphs of small diameter reach B within a few iterations:
// R-MAT-24 (p = 7) iterations 4, 5 and 6 take 1.6, 0.9 and 0.4 ms instead of 7.9, 7.9 and 4.5; the
// rule alone took its run from 40.1 to 24.2 ms and R-MAT-20's (p = 8) from 4.7 to 3.3.  One bound
// has to fit all: a component of three nodes or more that holds a register's maximum keeps the
// others below B, and then nothing is saved.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "hb_device.h"
#include "hb_kernels.h"
#include "hb_union.h"

namespace hb {

static constexpr int kBlock = 256;


// block-wide sums of per-lane counters, one atomic per counter per block, into the copy of
// the counters the block's number selects; k_finalize adds the copies up.  With one copy
// thousands of blocks end on the same few words, one after another: with 16, the k-mer run
// of 64 iterations takes 21.2 ms instead of 23.7, R-MAT-20's (p = 8) 2.88 instead of 3.31.
__device__ __forceinline__ void block_add(unsigned long long inc, unsigned long long arcs, unsigned long long nodes,
                                          unsigned long long chg, unsigned long long gathered,
                                          unsigned long long sat, const HbDev &d, int slot)
{
    constexpr int kWaves = kBlock / HB_WAVE;
    __shared__ unsigned long long red[6][kWaves];
    unsigned long long v[6] = {inc, arcs, nodes, chg, gathered, sat};
#pragma unroll
    for (int s = 1; s < HB_WAVE; s <<= 1)
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] += __shfl_xor(v[k], s);
    const int w = threadIdx.x / HB_WAVE;
    if ((threadIdx.x & (HB_WAVE - 1)) == 0)
#pragma unroll
        for (int k = 0; k < 6; ++k) red[k][w] = v[k];
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned long long t = 0;
        for (int i = 0; i < kWaves; ++i) t += red[threadIdx.x][i];
        const uint32_t at = threadIdx.x < 5 ? threadIdx.x * HB_NSLOT + slot : 5 * HB_NSLOT;
        if (t) atomicAdd(d.counts + (blockIdx.x % HB_COUNT_COPIES) * HB_COUNT_STRIDE + at, t);
    }
}

// f64 accumulation without contraction (hyper_ball.rs:823-825)
__device__ __forceinline__ bool accumulate(const HbDev &d, uint32_t u, float prev, float curr,
                                           double t, double inv_t)
{
    const float d32 = __fsub_rn(curr, prev);
    const double diff = (double)d32;
    if (diff > 0.0) {
        d.dist[u] = __dadd_rn(d.dist[u], __dmul_rn(t, diff));
        d.inv[u] = __dadd_rn(d.inv[u], __dmul_rn(inv_t, diff));
        return true;
    }
    return false;
}

// ---------------------------------------------------------------------------
// init: c_0(u) = {insert(u)} (hyper_ball.rs:716-721); est, accumulators
// ---------------------------------------------------------------------------
template <int P>
__global__ __launch_bounds__(kBlock) void k_init(HbDev d)
{
    // One thread per node computes the node's insertion (one SipHash-1-3 per node); the
    // wavefront then writes the rows of its 64 nodes, G lanes per row and 64 / G rows per
    // store, taking each row's insertion by shuffle, so the stores stay coalesced.
    constexpr uint32_t M = 1u << P, G = M / 16, RPI = HB_WAVE / G;
    const uint32_t lane = threadIdx.x % HB_WAVE, cl = lane % G;
    const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t first = u - lane;  // the wavefront's first node
    uint32_t word = 0;                // rank | idx << 8 | (no neighbours) << 31
    __shared__ uint32_t s_max[M];     // the block's share of the bound of all sketches
    if (d.sat_max) {
        for (uint32_t i = threadIdx.x; i < M; i += kBlock) s_max[i] = 0u;
        __syncthreads();
    }
    if (u < d.n) {
        uint32_t idx, rank;
        hb_index_rank(d.node_id ? d.node_id[u] : (uint32_t)u, P, &idx, &rank);
        const uint32_t e0 = d.off[u], deg = d.off[u + 1] - e0;
        word = rank | (idx << 8) | (deg == 0 ? 1u << 31 : 0u);
        // On a symmetric graph a node without neighbours and a pair of nodes that only have
        // each other reach no other sketch; leaving them out lets the giant component of a
        // random graph, which seldom lacks other nodes, attain the bound.
        if (d.sat_max) {
            const uint32_t w = d.sym && deg == 1 ? d.nbr[e0] : 0u;
            const bool alone = d.sym && (deg == 0 || (deg == 1 && d.off[w + 1] - d.off[w] == 1));
            if (!alone) atomicMax(s_max + idx, rank);
        }
    }
    if (d.sat_max) {  // one look per register and block; few blocks still raise one
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < M; i += kBlock)
            if (s_max[i] > d.sat_max[i]) atomicMax(d.sat_max + i, s_max[i]);
    }
#pragma unroll
    for (uint32_t k = 0; k < G; ++k) {
        const uint32_t r = k * RPI + lane / G;  // this store's row among the wavefront's nodes
        const uint32_t w = (uint32_t)__shfl((int)word, (int)r);
        const uint64_t node = first + r;
        if (node < d.n) {
            const uint32_t idx = (w >> 8) & 0xffffu, rank = w & 0xffu;
            uint32_t q[4] = {0, 0, 0, 0};
            if (idx / 16 == cl) q[(idx % 16) / 4] = rank << (8 * (idx % 4));
            const uint4 row = make_uint4(q[0], q[1], q[2], q[3]);
            *(uint4 *)(d.regs0 + (node << P) + cl * 16) = row;
            // a node without neighbours keeps c_0 forever and is never scheduled: both buffers
            if (w >> 31) *(uint4 *)(d.regs1 + (node << P) + cl * 16) = row;
        }
    }
    if (u < d.n) {
        // c_0 holds one register of rank >= 1 and m - 1 empty ones, so the estimator returns
        // linear counting of m - 1 zeros (launch_init checks that the HLL++ threshold admits it)
        d.est[u] = d.lc[M - 1];
        d.dist[u] = 0.0;
        d.inv[u] = 0.0;
    }
}

__global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t *p, uint64_t count, uint32_t value)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

// start of a run: its bitmaps and counters cleared, its state as of iteration 1
__global__ __launch_bounds__(kBlock) void k_start(HbIterState *st, HbIterState st0, uint32_t *p, uint64_t count)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *st = st0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

// ---------------------------------------------------------------------------
// push iterations (symmetric graph, few changes at t-1): u must be recomputed
// iff one of its neighbours changed, i.e. iff u is a neighbour of a changed node.
// k_begin sets those bits from the changed nodes' lists (a wavefront per bitmap
// word); k_push_compact lists them per degree bin with wavefront-aggregated appends
// and copies c_{t-1}(u) into the output buffer for every non-hub node that changed
// at t-1 but has no changed neighbour (hubs: k_merge copies).
// ---------------------------------------------------------------------------
// Start of iteration t: clear the bitmap iteration t writes (bits[t & 1]) and, where
// push iterations can occur, the active bitmap of iteration t + 1; carry the saturated
// nodes over; clear this iteration's ring record; in a push iteration also clear the per-bin list counts and
// mark this iteration's active bitmap.  The marking reads bits[(t - 1) & 1] and writes
// hb_active(t), neither of which the clearing touches.
__global__ __launch_bounds__(kBlock) void k_begin(HbDev d, uint32_t words)
{
    const HbIterState *st = d.st;
    if (st->done) return;
    const uint32_t it = st->iter;
    uint32_t *bw = (it & 1u) ? d.bits1 : d.bits0;
    const bool push = st->push != 0;
    if (push && blockIdx.x == 0 && threadIdx.x < 3) d.dyn_count[threadIdx.x] = 0u;
    if (blockIdx.x == 0 && threadIdx.x == 0) {  // this iteration's record
        d.rec->nf_lo = d.rec->nf_hi = 0ull;
        d.rec->push = push ? 1ull : 0ull;
    }
    uint32_t *next_active = d.active ? hb_active(d, it + 1) : nullptr;
    uint32_t *sat = d.sat_max ? hb_saturated(d, it) : nullptr;
    const uint32_t *sat_prev = d.sat_max ? hb_saturated(d, it - 1) : nullptr;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) {
        bw[i] = 0u;
        if (next_active) next_active[i] = 0u;
        if (sat) sat[i] = sat_prev[i];
    }
    if (!push) return;
    uint32_t *act = hb_active(d, it);
    const uint32_t *bitsR = (it & 1u) ? d.bits0 : d.bits1;
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    const uint32_t waves = gridDim.x * (kBlock / HB_WAVE);
    for (uint32_t wd = blockIdx.x * (kBlock / HB_WAVE) + threadIdx.x / HB_WAVE; wd < words; wd += waves) {
        uint32_t m = bitsR[wd];  // one word per wavefront: the loop below is uniform
        while (m) {
            const uint32_t w = wd * 32u + (uint32_t)(__ffs(m) - 1);
            m &= m - 1u;
            const uint32_t e1 = d.off[w + 1];
            for (uint32_t e = d.off[w] + lane; e < e1; e += HB_WAVE) {
                const uint32_t u = d.nbr[e], bit = 1u << (u & 31u);
                if (!(act[u >> 5] & bit)) atomicOr(act + (u >> 5), bit);
            }
        }
    }
}

template <int P>
__global__ __launch_bounds__(kBlock) void k_push_compact(HbDev d, uint32_t words)
{
    const HbIterState *st = d.st;
    if (st->done || !st->push) return;
    const uint32_t *bitsR = (st->iter & 1u) ? d.bits0 : d.bits1;
    const uint8_t *in = st->parity ? d.regs1 : d.regs0;
    uint8_t *out = st->parity ? d.regs0 : d.regs1;
    const uint32_t *act = hb_active(d, st->iter);
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    // the trip count is uniform across a wavefront, so every lane takes part in the ballots
    for (uint32_t base = blockIdx.x * blockDim.x; base < words; base += gridDim.x * blockDim.x) {
        const uint32_t wd = base + threadIdx.x;
        uint32_t a = 0, c = 0;
        if (wd < words) {
            a = act[wd];
            c = bitsR[wd] & ~a;
        }
        while (c) {
            const uint32_t u = wd * 32u + (uint32_t)(__ffs(c) - 1);
            c &= c - 1u;
            if (d.off[u + 1] - d.off[u] > d.wave_max) continue;
            const uint4 *src = (const uint4 *)(in + ((uint64_t)u << P));
            uint4 *dst = (uint4 *)(out + ((uint64_t)u << P));
#pragma unroll
            for (int k = 0; k < (1 << P) / 16; ++k) dst[k] = src[k];
        }
        while (__ballot(a != 0u)) {
            uint32_t u = 0, bin = 3;
            if (a) {
                u = wd * 32u + (uint32_t)(__ffs(a) - 1);
                a &= a - 1u;
                const uint32_t deg = d.off[u + 1] - d.off[u];
                // hubs (bin 3) are not listed: k_chunk / k_merge check their own chunks;
                // deg 0 cannot occur on a symmetric graph and is never listed either
                bin = deg == 0 ? 3u : deg <= d.small_max ? 0u : deg <= d.mid_max ? 1u : deg <= d.wave_max ? 2u : 3u;
            }
            for (uint32_t b = 0; b < 3; ++b) {
                const unsigned long long m = __ballot(bin == b);
                if (!m) continue;
                const int leader = __ffsll(m) - 1;
                uint32_t pos = 0;
                if ((int)lane == leader) pos = atomicAdd(d.dyn_count + b, (uint32_t)__popcll(m));
                pos = __shfl(pos, leader);
                if (bin == b)
                    d.dyn_list[d.dyn_base[b] + pos + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = u;
            }
        }
    }
}

// Order-free fingerprints of the arc multiset and of its reverse, with h a
// splitmix64 mix of the pair: acc[0] = sum h(u, v), acc[1] = sum h(v, u),
// acc[2] = sum h(u, v)^2, acc[3] = sum h(v, u)^2 (wrapping).  A symmetric multiset
// gives acc[0] == acc[1] and acc[2] == acc[3]; any other CSR matches both sums only
// by a coincidence of two 64-bit equations.
__device__ __forceinline__ uint64_t hb_mix64(uint64_t z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

// Each block writes its four sums to part[4 * block]; sum_columns adds the blocks.
__device__ __forceinline__ void hb_fp_add(unsigned long long *a, uint64_t u, uint64_t v)
{
    const uint64_t hf = hb_mix64((u << 32) | v), hb = hb_mix64((v << 32) | u);
    a[0] += hf;
    a[1] += hb;
    a[2] += hf * hf;
    a[3] += hb * hb;
}

// A wavefront takes kFpArcs * 64 consecutive arcs at a time, loaded coalesced into its lanes'
// registers.  Their tails: a 64-way search over the offsets finds the first one's, the
// offsets that follow, read coalesced, put each node's id where its arcs start in LDS, and a
// running maximum spreads the ids over the arcs (each lane over a run of kFpArcs, a scan over
// the lanes joining the runs; one pad word per run keeps LDS free of bank conflicts).  Hubs
// and runs of empty nodes cost no more than other arcs and nodes.  When each lane read and
// walked kFpArcs = 32 arcs of its own, 128 bytes from the next lane's, 16M arcs took 583 us, 31M
// 688, a graph of 4k nodes 24; now 77, 139 and 12 (kFpArcs of 16: 130 and 169, of 4: 77 and 130).
constexpr uint32_t kFpArcs = 8;

__global__ __launch_bounds__(kBlock) void k_arc_fingerprint(const uint32_t *off, const uint32_t *nbr, uint32_t n,
                                                            uint64_t arcs, unsigned long long *part)
{
    constexpr uint32_t kSpan = kFpArcs * HB_WAVE, kRun = kFpArcs + 1;
    __shared__ unsigned long long red[kBlock / HB_WAVE][4];
    __shared__ uint32_t s_tail[kBlock / HB_WAVE][HB_WAVE * kRun];
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1), wv = threadIdx.x / HB_WAVE;
    uint32_t *tail = s_tail[wv];
    unsigned long long a[4] = {0, 0, 0, 0};
    const uint64_t step = (uint64_t)gridDim.x * (kBlock / HB_WAVE) * kSpan;
    for (uint64_t base = ((uint64_t)blockIdx.x * (kBlock / HB_WAVE) + wv) * kSpan; base < arcs; base += step) {
        const uint32_t span = (uint32_t)min<uint64_t>(kSpan, arcs - base);
        uint32_t x[kFpArcs], run[kFpArcs];
#pragma unroll
        for (uint32_t k = 0; k < kFpArcs; ++k) {
            const uint32_t i = k * HB_WAVE + lane;
            x[k] = i < span ? nbr[base + i] : 0u;
            tail[lane * kRun + k] = 0u;
        }
        uint32_t lo = 0, len = n;  // the largest u with off[u] <= base is one of lo .. lo + len - 1
        while (len > 1) {
            const uint32_t stride = (len + HB_WAVE - 1) / HB_WAVE;
            const uint64_t i = (uint64_t)lane * stride;
            const unsigned long long m = __ballot(i < len && off[lo + i] <= base);
            const uint32_t c = (uint32_t)__popcll(m) - 1u;  // off[lo] <= base
            lo += c * stride;
            len = min(stride, len - c * stride);
        }
        __builtin_amdgcn_wave_barrier();  // the zeros are written
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (uint32_t u0 = lo + 1;; u0 += HB_WAVE) {
            const uint32_t u = u0 + lane;
            const uint64_t start = u < n ? off[u] : arcs;
            const bool in = start < base + span;
            if (in && off[u + 1] != start) {
                const uint32_t i = (uint32_t)(start - base);
                tail[i + i / kFpArcs] = u;
            }
            if (__ballot(!in)) break;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t top = lane == 0 ? lo : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kFpArcs; ++k) run[k] = top = max(top, tail[lane * kRun + k]);
        for (int o = 1; o < HB_WAVE; o <<= 1) {
            const uint32_t below = __shfl_up(top, o);
            if (lane >= (uint32_t)o) top = max(top, below);
        }
        const uint32_t before = __shfl_up(top, 1);
#pragma unroll
        for (uint32_t k = 0; k < kFpArcs; ++k) tail[lane * kRun + k] = lane ? max(run[k], before) : run[k];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (uint32_t k = 0; k < kFpArcs; ++k) {
            const uint32_t i = k * HB_WAVE + lane;
            if (i < span) hb_fp_add(a, tail[i + i / kFpArcs], x[k]);
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read the tails
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    for (int k = 0; k < 4; ++k)
        for (int o = 1; o < HB_WAVE; o <<= 1) a[k] += __shfl_xor(a[k], o);
    if (lane == 0)
        for (int k = 0; k < 4; ++k) red[wv][k] = a[k];
    __syncthreads();
    if (threadIdx.x < 4) {
        unsigned long long sum = 0;
        for (int w = 0; w < kBlock / HB_WAVE; ++w) sum += red[w][threadIdx.x];
        part[4 * blockIdx.x + threadIdx.x] = sum;
    }
}

// ---------------------------------------------------------------------------
// dense iterations of an id-range bin in the chain layout at p = 5 or 6: one lane per
// node, its whole 2^p-byte row in the lane's registers (W = 2^p / 16 words)
// ---------------------------------------------------------------------------
// With a team of G = 2^p / 16 lanes per node (union_node_window) a wavefront holds 16
// nodes at p = 6, and the lanes of a team repeat each other's per-node work: offsets,
// addresses, the estimate.  On a graph of long low-degree chains that union is bound by
// each node's chain of dependent memory accesses, not by bytes, so what counts is how
// many nodes are in flight.  Here a wavefront holds 64 consecutive nodes lo..lo+63:
//   1. their rows c_{t-1} enter the wavefront's LDS window by coalesced 16-byte loads;
//   2. each lane takes its node's row from the window and merges its neighbours' rows,
//      from the window when the neighbour is one of the 64, else from memory;
//   3. the new rows go back through the window and out by coalesced stores;
//   4. estimate and accumulators per lane; the changed bits of the 64 nodes are ORed
//      into the bitmap with one atomic per 32-bit word.
// Same registers, estimates and accumulators as union_node.

// an iteration whose id-range bins k_union_rows runs instead of k_union: dense (no
// frontier gathers, no push list).  That includes the first: k_init wrote every node's
// c_0 row into the buffer iteration 1 reads, and gathering those rows, most of them from
// the LDS window, is cheaper here than hashing every neighbour id as k_union does.
__device__ __forceinline__ bool rows_iteration(const HbDev &d, const HbIterState &st)
{
    return !st.push && (st.iter == 1 || !(d.frontier && !st.skip_scan));
}

// The window of a wavefront is W planes of 64 uint4: plane q holds chunk q (bytes
// 16q .. 16q + 15) of the 64 rows, row w at position w ^ row_perm(q).  The permutation
// keeps a wavefront's structured accesses free of LDS bank conflicts: a lane reading
// chunk q of its own row, and the coalesced copies (chunk q of rows 64/W apart per
// lane group), land in distinct 16-byte bank groups for 8 and for 16 lanes per cycle.
template <int W>
__device__ __forceinline__ uint32_t row_perm(uint32_t q)
{
    return W == 4 ? (0xCA60u >> (4 * q)) & 15u : (0xC0u >> (4 * q)) & 15u;  // {0,6,10,12} / {0,12}
}

template <int W>
__device__ __forceinline__ uint32_t win_index(uint32_t w, uint32_t q)
{
    return q * HB_WAVE + (w ^ row_perm<W>(q));
}

// row c_{t-1}(x): from the window when x is one of its nodes lo .. lo + span - 1
template <int P>
__device__ __forceinline__ void row_fetch(uint4 *r, uint32_t x, uint32_t lo, uint32_t span, const uint4 *win,
                                          const uint8_t *__restrict__ in)
{
    constexpr int W = (1 << P) / 16;
    if (x - lo < span) {
#pragma unroll
        for (int q = 0; q < W; ++q) r[q] = win[win_index<W>(x - lo, q)];
    } else {
        const uint4 *g = (const uint4 *)(in + ((uint64_t)x << P));
#pragma unroll
        for (int q = 0; q < W; ++q) r[q] = g[q];
    }
}

// Seven wavefronts per SIMD (71 VGPRs at p = 6, no spill): 448 nodes in flight per SIMD
// against 128 for union_node_window at eight wavefronts of 16.  On the k-mer graph (p = 6) a
// launch takes 0.362 ms against 0.583 for union_node_window; at eight (64 VGPRs, spills
// outside the node loop only) 0.365 ms.  Since the iteration counters have copies 0.294 ms, with
// the rows written as streaming data 0.282: 1.38 GB at 4.9 TB/s, where a copy reaches 5.2 to 6.
// The bin's base must be a multiple of 64.
template <int P>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_union_rows(
    HbDev d, uint32_t base, uint32_t count, int slot_id)
{
    constexpr int W = (1 << P) / 16;
    static_assert(W == 2 || W == 4, "p = 5 or 6");
    const HbIterState *st = d.st;
    if (st->done || !rows_iteration(d, *st)) return;
    HB_TABLES_LDS(P, d, tb)
    __shared__ uint4 s_win[kBlock * W];  // 64 rows per wavefront
    const uint32_t it = st->iter;
    const uint32_t lane = threadIdx.x % HB_WAVE;
    uint4 *win = s_win + (threadIdx.x / HB_WAVE) * (HB_WAVE * W);
    HbView v{};
    v.in = st->parity ? d.regs1 : d.regs0;
    v.out = st->parity ? d.regs0 : d.regs1;
    v.dist = d.dist;
    v.inv = d.inv;
    v.t = st->t;
    v.inv_t = st->inv_t;
    const uint8_t *__restrict__ in = v.in;
    const uint32_t *__restrict__ nb = d.nbr;
    uint32_t *bitsW = (it & 1u) ? d.bits1 : d.bits0;
    // chunk r * 64 + lane of the wavefront's rows (a coalesced copy) is chunk lane % W of
    // row r * 64 / W + lane / W, at window index cidx + r * 64 / W (the permutation only
    // touches the low 4 bits of a row, below 64 / W)
    constexpr uint32_t RPC = HB_WAVE / W;  // rows per coalesced copy instruction
    const uint32_t lw = lane / W;
    const uint32_t cidx = win_index<W>(lw, lane % W);
    unsigned long long n_inc = 0, n_arcs = 0, n_nodes = 0, n_chg = 0;  // the wavefront's counts
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / HB_WAVE);
    const uint32_t stride = __builtin_amdgcn_readfirstlane(gridDim.x) * kBlock;
    for (uint32_t w0 = (blockIdx.x * (kBlock / HB_WAVE) + wave) * HB_WAVE; w0 < count; w0 += stride) {
        const uint32_t lo = base + w0, span = min((uint32_t)HB_WAVE, count - w0);
        const bool valid = lane < span;
        const uint32_t u = lo + lane;
        uint32_t e0 = 0, e1 = 0;
        float prev = 0.0f;
        if (valid) {
            e0 = d.off[u];
            e1 = d.off[u + 1];
            prev = d.est[u];
        }
        const uint4 *src = (const uint4 *)(in + ((uint64_t)lo << P));
#pragma unroll
        for (int r = 0; r < W; ++r)
            if ((int)lw < (int)span - r * (int)RPC) win[cidx + r * RPC] = src[r * HB_WAVE + lane];
        // LDS operations of one wavefront complete in order; the barrier and fence keep
        // the compiler from moving window accesses across each other
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint4 acc[W];
#pragma unroll
        for (int q = 0; q < W; ++q) acc[q] = valid ? win[win_index<W>(lane, q)] : make_uint4(0, 0, 0, 0);
        uint32_t e = e0;
        for (; e < e1; ++e) {
            uint4 r0[W];
            row_fetch<P>(r0, nb[e], lo, span, win, in);
#pragma unroll
            for (int q = 0; q < W; ++q) acc[q] = hb_bmax4(acc[q], r0[q]);
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read the window
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t diffw = 0;
#pragma unroll
        for (int q = 0; q < W; ++q) {
            const uint4 o = win[win_index<W>(lane, q)];
            diffw |= (acc[q].x != o.x) | (acc[q].y != o.y) | (acc[q].z != o.z) | (acc[q].w != o.w);
            win[win_index<W>(lane, q)] = acc[q];
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint4 *dst = (uint4 *)(v.out + ((uint64_t)lo << P));
#pragma unroll
        for (int r = 0; r < W; ++r)
            if ((int)lw < (int)span - r * (int)RPC) store_row(dst + r * HB_WAVE + lane, win[cidx + r * RPC]);
        // counts: nodes lo .. lo + span - 1 hold arcs off[lo] .. off[lo + span] - 1
        n_nodes += span;
        n_arcs += (uint32_t)__builtin_amdgcn_readlane((int)e1, (int)span - 1) -
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)e0);
        const float curr = hb_estimate_row<W>(tb, acc);
        const bool changed = valid && diffw != 0;
        bool inc = false;
        if (valid) {
            inc = accumulate(v, u, prev, curr);  // reads the accumulators only if they change
            d.est[u] = curr;
        }
        n_inc += __popcll(__ballot(inc));
        // the changed bits of nodes lo .. lo + 63 (lo a multiple of 64): two bitmap words,
        // ORed atomically since the last may also hold bits of nodes past the bin
        const unsigned long long mask = __ballot(changed);
        n_chg += __popcll(mask);
        const uint32_t bits_lo = (uint32_t)mask, bits_hi = (uint32_t)(mask >> 32);
        if (lane == 0 && bits_lo) atomicOr(bitsW + (lo >> 5), bits_lo);
        if (lane == 1 && bits_hi) atomicOr(bitsW + (lo >> 5) + 1, bits_hi);
        // the next trip's window writes follow this trip's reads
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    const bool first_lane = lane == 0;
    block_add(first_lane ? n_inc : 0, first_lane ? n_arcs : 0, first_lane ? n_nodes : 0, first_lane ? n_chg : 0,
              first_lane ? n_arcs : 0, 0, d, slot_id);
}

// the bound of all sketches, packed as registers are, into LDS (2^P bytes at s)
template <int P>
__device__ __forceinline__ void stage_bound(const HbDev &d, uint32_t *s)
{
    for (uint32_t i = threadIdx.x; i < (1u << P) / 4; i += kBlock) {
        const uint4 r = *(const uint4 *)(d.sat_max + 4 * i);
        s[i] = r.x | (r.y << 8) | (r.z << 16) | (r.w << 24);
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// union over the neighbours of listed nodes; a team of T lanes per node
// (T = G: one sketch copy; T > G: S = T/G copies split the neighbours)
// ---------------------------------------------------------------------------
// Wavefronts per SIMD: the gathers are latency-bound, so more wavefronts in flight help until
// the register bound makes the compiler spill.  8 (at most 64 VGPRs) took the k-mer graph
// (p = 6, four-lane teams in the degree layout) from 59.5 to 49.5 ms per run.  The one-copy
// bins run at 7: at 8, with the saturation checks, they spill 36 VGPRs and R-MAT-24's dense
// iterations (p = 7) take 8.13 ms against 7.97 at 7 and 8.02 at 6.  The teams of 32 and 64
// lanes run at 6 at p >= 7 (80 VGPRs, no spill).  The k-mer graph's dense iterations run
// k_union_rows instead.
template <int P, int T, bool kFirst>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(P >= 7 && T >= 32 ? 6 : T == (1 << P) / 16 ? 7 : 8))) void k_union(
    HbDev d, const uint32_t *__restrict__ list, uint32_t base, uint32_t count, int slot_id)
{
    const HbIterState *st = d.st;
    if (st->done) return;
    if constexpr (!kFirst && T == (1 << P) / 16 && (P == 5 || P == 6))
        if (d.rows && !list && (base & 63u) == 0 && rows_iteration(d, *st)) return;  // k_union_rows runs it
    const uint32_t it = st->iter;
    if (st->push) {  // only the bin's nodes with a changed neighbour (k_push_compact)
        list = d.dyn_list + d.dyn_base[slot_id];
        count = d.dyn_count[slot_id];
    }
    if (blockIdx.x * (kBlock / T) >= count) return;  // most blocks of a push iteration
    HB_TABLES_LDS(P, d, tb)
    HbView v;
    v.off = d.off;
    v.nbr = d.nbr;
    v.orig = d.orig;
    v.node_id = d.node_id;
    v.in = st->parity ? d.regs1 : d.regs0;
    v.out = st->parity ? d.regs0 : d.regs1;
    v.est = d.est;
    v.dist = d.dist;
    v.inv = d.inv;
    v.bitsR = (it & 1u) ? d.bits0 : d.bits1;
    v.bitsW = (it & 1u) ? d.bits1 : d.bits0;
    v.t = st->t;
    v.inv_t = st->inv_t;
    v.use_frontier = d.frontier && it > 1 && !st->skip_scan && !st->push;
    // outside dense iterations only the neighbours that changed at t-1 are gathered
    v.gather_bits = d.frontier && it > 1 && !st->skip_scan ? v.bitsR : nullptr;
    // iteration 1's register arrays (16 u32 per lane), the LDS window of the chain layout's
    // dense iterations (one uint4 per lane) or the bound of all sketches (2^P bytes)
    constexpr uint32_t kScratch = kFirst ? kBlock * 16 : T == (1 << P) / 16 ? kBlock * 4 : (1 << P) / 4;
    __shared__ __attribute__((aligned(16))) uint32_t s_scr[kScratch];
    static_assert(kScratch >= (1 << P) / 4, "room for the bound");
    v.scr = s_scr;
    v.sym = d.sym != 0;
    if (!kFirst && d.sat_max) {
        stage_bound<P>(d, s_scr);
        v.satR = hb_saturated(d, it - 1);
        v.satW = hb_saturated(d, it);
        v.bound = reinterpret_cast<const uint4 *>(s_scr);
        v.sat_scan = st->sat_scan != 0;
    }
    const uint32_t tl = threadIdx.x % T;
    const uint32_t teams_per_grid = gridDim.x * (kBlock / T);
    HbCounts c;
    if constexpr (!kFirst && T == (1 << P) / 16 && P != 5 && P != 6) {
        // dense iteration over an id-range bin: each wavefront's teams hold consecutive
        // nodes, and neighbours among them come from the wavefront's LDS window (at p = 5
        // and 6 k_union_rows runs these iterations)
        if (d.window && !list && !v.gather_bits) {
            uint4 *win = reinterpret_cast<uint4 *>(s_scr) + (threadIdx.x / HB_WAVE) * HB_WAVE;
            const uint32_t in_wave = (threadIdx.x % HB_WAVE) / T;
            for (uint32_t team = blockIdx.x * (kBlock / T) + threadIdx.x / T; team < count; team += teams_per_grid) {
                const uint32_t lo = base + team - in_wave;
                union_node_window<P, T>(v, tb, base + team, tl, c, lo, min(lo + HB_WAVE / T, base + count), win);
            }
            block_add(c.inc, c.arcs, c.nodes, c.chg, c.gathered, c.sat, d, slot_id);
            return;
        }
    }
    auto run = [&](auto gather) {
        constexpr Gather kGather = decltype(gather)::value;
        if (list) {
            for (uint32_t team = blockIdx.x * (kBlock / T) + threadIdx.x / T; team < count; team += teams_per_grid) {
                const uint32_t u = list[team];
                const uint32_t r = union_node<P, T, kGather>(v, tb, u, tl, c);
                if (tl == 0 && (r & kChangedBit)) bit_set(v.bitsW, u);
                if (tl == 0 && (r & kSaturatedBit)) bit_set(v.satW, u);
            }
        } else {
            const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / HB_WAVE);
            for (uint32_t t0 = blockIdx.x * (kBlock / T) + wave * (HB_WAVE / T); t0 < count; t0 += teams_per_grid)
                union_wave<P, T, kGather>(v, tb, base + t0, count - t0, c);
        }
    };
    if constexpr (kFirst) run(std::integral_constant<Gather, Gather::kFirst>{});
    else if (v.gather_bits) run(std::integral_constant<Gather, Gather::kChanged>{});
    else run(std::integral_constant<Gather, Gather::kAll>{});
    block_add(c.inc, c.arcs, c.nodes, c.chg, c.gathered, c.sat, d, slot_id);
}

// ---------------------------------------------------------------------------
// hubs, phase 1: one wavefront per chunk of a hub's neighbour list writes the
// chunk's partial union to scratch (not the hub's own registers)
// ---------------------------------------------------------------------------
template <int P, bool kFirst>
__global__ __launch_bounds__(kBlock) void k_chunk(HbDev d, const uint32_t *__restrict__ tnode,
                                                  const uint32_t *__restrict__ tbeg,
                                                  const uint32_t *__restrict__ tend, uint32_t ntasks)
{
    constexpr uint32_t M = 1u << P, G = M / 16, T = HB_WAVE, S = T / G;
    const HbIterState *st = d.st;
    if (st->done) return;
    const uint32_t it = st->iter;
    const uint8_t *__restrict__ in = st->parity ? d.regs1 : d.regs0;
    const uint32_t *__restrict__ bitsR = (it & 1u) ? d.bits0 : d.bits1;
    const bool use_frontier = d.frontier && it > 1 && !st->skip_scan;
    // push iteration: a hub whose active bit is clear has no changed neighbour at all
    const bool push = st->push != 0;
    __shared__ __attribute__((aligned(16))) uint32_t s_scr[kFirst ? kBlock * 16 : M / 4];  // as in k_union
    const uint32_t tl = threadIdx.x % T, cl = tl % G, slot = tl / G;
    const uint32_t waves_per_grid = gridDim.x * (kBlock / T);
    unsigned long long c_arcs = 0, c_gathered = 0;
    const uint32_t *satR = nullptr;
    const uint4 *bound = reinterpret_cast<const uint4 *>(s_scr);
    if (!kFirst && d.sat_max) {
        stage_bound<P>(d, s_scr);
        satR = hb_saturated(d, it - 1);
    }
    const bool sat_scan = satR && st->sat_scan;

    for (uint32_t task = blockIdx.x * (kBlock / T) + threadIdx.x / T; task < ntasks;
         task += waves_per_grid) {
        const uint32_t eb = tbeg[task], ee = tend[task];
        const uint32_t *__restrict__ nb = d.nbr + eb;
        const uint32_t *__restrict__ nbh = d.orig + eb;
        const uint32_t len = ee - eb;
        bool active = !(push && !bit_test(hb_active(d, it), tnode[task])) && !(satR && bit_test(satR, tnode[task]));
        uint32_t scanned = 0;
        const bool sat = active && sat_scan && sat_neighbour<T>(satR, nb, len, tl, scanned);
        if (use_frontier && active && !sat) {
            uint32_t any = 0;
            for (uint32_t j = tl; j < len; j += T) any |= bit_test(bitsR, nb[j]);
            active = hb_copy_or<T>(any) != 0;
        }
        if (tl == 0) d.chunk_flag[task] = active ? 1u : 0u;
        if (!active) continue;
        if (sat) {  // the hub becomes the bound through this chunk
            if (slot == 0) *(uint4 *)(d.scratch + ((uint64_t)task << P) + cl * 16) = bound[cl];
            if (tl == 0) c_arcs += scanned;
            continue;
        }
        uint32_t gathered = 0;  // by this lane's copy
        const uint4 none = make_uint4(0, 0, 0, 0);
        uint4 acc;
        if constexpr (kFirst)
            acc = hb_gather_union<P, S, Gather::kFirst>(in, s_scr, nullptr, nb, nbh, len, slot, cl, none, gathered);
        else
            acc = use_frontier
                      ? hb_gather_union<P, S, Gather::kChanged>(in, nullptr, bitsR, nb, nbh, len, slot, cl, none, gathered)
                      : hb_gather_union<P, S, Gather::kAll>(in, nullptr, nullptr, nb, nbh, len, slot, cl, none, gathered);
        if (cl == 0) c_gathered += gathered;
#pragma unroll
        for (uint32_t s = G; s < T; s <<= 1) acc = hb_bmax4(acc, hb_shfl_xor4<T>(acc, s));
        if (slot == 0) *(uint4 *)(d.scratch + ((uint64_t)task << P) + cl * 16) = acc;
        if (tl == 0) c_arcs += len;
    }
    block_add(0, c_arcs, 0, 0, c_gathered, 0, d, HB_SLOT_CHUNK);
}

// hubs, phase 2: one wavefront per hub merges its own registers with the
// partials of its recomputed chunks (a chunk that was not recomputed has no
// changed neighbour, so its union is already contained in c_{t-1}(u))
template <int P>
__global__ __launch_bounds__(kBlock) void k_merge(HbDev d, const uint32_t *__restrict__ hnode,
                                                  const uint32_t *__restrict__ htask0,
                                                  const uint32_t *__restrict__ hntask, uint32_t nhubs)
{
    constexpr uint32_t M = 1u << P, G = M / 16, T = HB_WAVE, S = T / G;
    const HbIterState *st = d.st;
    if (st->done) return;
    HB_TABLES_LDS(P, d, tb)
    const uint32_t it = st->iter;
    const double t = st->t, inv_t = st->inv_t;
    const uint8_t *__restrict__ in = st->parity ? d.regs1 : d.regs0;
    uint8_t *__restrict__ out = st->parity ? d.regs0 : d.regs1;
    const uint32_t *__restrict__ bitsR = (it & 1u) ? d.bits0 : d.bits1;
    uint32_t *bitsW = (it & 1u) ? d.bits1 : d.bits0;
    const uint32_t tl = threadIdx.x % T, cl = tl % G, slot = tl / G;
    const uint32_t waves_per_grid = gridDim.x * (kBlock / T);
    unsigned long long c_inc = 0, c_nodes = 0, c_chg = 0, c_sat = 0;
    __shared__ __attribute__((aligned(16))) uint32_t s_bound[M / 4];
    const bool sat = d.sat_max && it > 1;
    if (sat) stage_bound<P>(d, s_bound);
    const uint4 *bound = reinterpret_cast<const uint4 *>(s_bound);

    for (uint32_t h = blockIdx.x * (kBlock / T) + threadIdx.x / T; h < nhubs; h += waves_per_grid) {
        const uint32_t u = hnode[h], t0 = htask0[h], nt = hntask[h];
        uint32_t any = 0;
        for (uint32_t j = tl; j < nt; j += T) any |= d.chunk_flag[t0 + j];
        const bool active = hb_copy_or<T>(any) != 0;
        if (!active) {
            if (slot == 0 && bit_test(bitsR, u))
                *(uint4 *)(out + ((uint64_t)u << P) + cl * 16) =
                    *(const uint4 *)(in + ((uint64_t)u << P) + cl * 16);
            continue;
        }
        const uint4 own = *(const uint4 *)(in + ((uint64_t)u << P) + cl * 16);
        uint4 acc = own;
        for (uint32_t j = slot; j < nt; j += S)
            if (d.chunk_flag[t0 + j])
                acc = hb_bmax4(acc, *(const uint4 *)(d.scratch + ((uint64_t)(t0 + j) << P) + cl * 16));
#pragma unroll
        for (uint32_t s = G; s < T; s <<= 1) acc = hb_bmax4(acc, hb_shfl_xor4<T>(acc, s));
        uint32_t diffw = (acc.x != own.x) | (acc.y != own.y) | (acc.z != own.z) | (acc.w != own.w);
        if (sat) {  // bit 1: a register is below the bound
            const uint4 f = bound[cl];
            diffw |= ((acc.x != f.x) | (acc.y != f.y) | (acc.z != f.z) | (acc.w != f.w)) << 1;
        }
        diffw = hb_copy_or<G>(diffw);
        const bool changed = (diffw & 1u) != 0;
        const float curr = hb_estimate_copy<G>(tb, acc);
        if (slot == 0) *(uint4 *)(out + ((uint64_t)u << P) + cl * 16) = acc;
        if (tl == 0) {
            const float prev = d.est[u];
            if (accumulate(d, u, prev, curr, t, inv_t)) c_inc += 1;
            d.est[u] = curr;
            if (sat && !(diffw & 2u)) {  // a hub has many neighbours: it is part of the bound
                atomicOr(hb_saturated(d, it) + (u >> 5), 1u << (u & 31u));
                c_sat += d.off[u + 1] - d.off[u];
            }
            if (changed) {
                atomicOr(bitsW + (u >> 5), 1u << (u & 31u));
                c_chg += 1;
            }
            c_nodes += 1;
        }
    }
    block_add(c_inc, 0, c_nodes, c_chg, 0, c_sat, d, HB_SLOT_MERGE);
}

// ---------------------------------------------------------------------------
// precisions 11..16: one wavefront per node, 64 lanes x 16 registers to a 1 KiB chunk of
// the row, up to four chunks at a time in registers (wider rows go in passes).  What bounds
// it is the rows it reads, so their loads are kept in flight eight at a time; long lists are
// cut into tasks whose partial rows the hub's wavefront then reads as if they were its
// neighbours'; iteration 1 hashes ids as at p <= 10; outside dense iterations only changed
// neighbours are read, and saturated nodes (HbDev::sat_max) nothing at all.
// De Bruijn graph (n = 16,384, 131,068 arcs, p = 12): its 8 iterations take 1.07 ms, a dense one
// 0.115 (0.67 GB of rows: 5.8 TB/s); 2.99 ms with a loop of single loads per chunk, an LDS
// histogram for the estimate and a serial replay of the sums that are not exact.  R-MAT-15
// (p = 13) 126 -> 3.7 ms, R-MAT-17 (p = 11) 47.9 -> 2.0 ms, where hubs were one wavefront's.
// Three wavefronts per SIMD (up to 161 VGPRs) beat four (126 and spills: 1.24 ms).
// ---------------------------------------------------------------------------
template <int P>
struct Wide {
    static constexpr uint32_t M = 1u << P;
    static constexpr int CHUNKS = M / 1024, CG = CHUNKS < 4 ? CHUNKS : 4, PASSES = CHUNKS / CG;
};

// Zeros, maximum and sum of a row's registers, per lane and then over the wavefront.  s24 =
// sum of 2^(24 - M) over the registers M <= 24: exact, and all of them unless mx > 24.
struct WideSum {
    uint32_t z = 0, mx = 0;
    unsigned long long s24 = 0;

    __device__ void add(uint4 a)
    {
        z += hb_zero_bytes(a.x) + hb_zero_bytes(a.y) + hb_zero_bytes(a.z) + hb_zero_bytes(a.w);
        mx = max(mx, hb_max_byte(hb_bmax(hb_bmax(a.x, a.y), hb_bmax(a.z, a.w))));
        uint32_t k = 0;  // 16 terms of at most 2^24
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int b = 0; b < 4; ++b) k += (1u << 24) >> min((w[q] >> (8 * b)) & 0xffu, 31u);
        s24 += k;
    }
    __device__ void reduce()
    {
#pragma unroll
        for (int o = 1; o < HB_WAVE; o <<= 1) {
            z += __shfl_xor(z, o);
            mx = max(mx, (uint32_t)__shfl_xor(mx, o));
            s24 += __shfl_xor(s24, o);
        }
    }
};

// S + the 16 registers of lane `from`, one f32 add each in register order
__device__ __forceinline__ float wide_replay16(float S, uint4 a, int from)
{
    const uint32_t w[4] = {(uint32_t)__builtin_amdgcn_readlane((int)a.x, from),
                           (uint32_t)__builtin_amdgcn_readlane((int)a.y, from),
                           (uint32_t)__builtin_amdgcn_readlane((int)a.z, from),
                           (uint32_t)__builtin_amdgcn_readlane((int)a.w, from)};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int b = 0; b < 4; ++b) S = __fadd_rn(S, hb_pow2neg((w[q] >> (8 * b)) & 0xffu));
    return S;
}

// The reference's sequential f32 sum of 2^-M over a row whose sum is not exact in f32
// (row(c): this lane's registers of chunk c).  Let the final sum lie below 2^(E+1).  A term of
// at least u = 2^(E-23) adds exactly to a running sum that is a multiple of u, in any order;
// only the few smaller terms (M > 23 - E) can round, and, once one of them has left bits
// below u in the sum, the adds that carry it into a higher binade.  So the wavefront adds
// whole lanes (16 registers each) by prefix sums, exact in f64, up to the next lane that
// holds such an add, and replays that lane add by add.  Rows with a register above 35, for
// which f64 would not be exact, are replayed throughout.
template <int CHUNKS, class Row>
__device__ float wide_sequential_sum(uint32_t mx, Row row)
{
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    auto lane_sum = [](uint4 a) {
        double g = 0.0;
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                g += __longlong_as_double((long long)(1023 - ((w[q] >> (8 * b)) & 0xffu)) << 52);
        return g;
    };
    float S = 0.0f;
    if (mx > 35) {
        for (int c = 0; c < CHUNKS; ++c) {
            const uint4 a = row(c);
            for (int l = 0; l < HB_WAVE; ++l) S = wide_replay16(S, a, l);
        }
        return S;
    }
    double total = 0.0;
    for (int c = 0; c < CHUNKS; ++c) total += lane_sum(row(c));
#pragma unroll
    for (int o = 1; o < HB_WAVE; o <<= 1) total += __shfl_xor(total, o);
    // no running sum exceeds the exact one by its rounding errors, 2^16 times 2^-24 of it
    const int E = (int)((__double_as_longlong(total * 1.01) >> 52) & 0x7ff) - 1023;
    const double per_u = __longlong_as_double((long long)(1023 - E + 23) << 52);
    const uint32_t thr = (uint32_t)max(23 - E, 0);
    for (int c = 0; c < CHUNKS; ++c) {
        const uint4 a = row(c);
        double X = lane_sum(a);
        const bool tiny = hb_max_byte(hb_bmax(hb_bmax(a.x, a.y), hb_bmax(a.z, a.w))) > thr;
#pragma unroll
        for (int o = 1; o < HB_WAVE; o <<= 1) {
            const double y = __shfl_up(X, o);
            if ((int)lane >= o) X += y;
        }
        uint32_t pos = 0;
        double before = 0.0;  // prefix sum of the lanes < pos
        while (pos < HB_WAVE) {
            const double s = (double)S, q = s * per_u;
            bool stop = tiny;
            if (q != floor(q)) {  // bits below u: the next binade rounds
                const double next = __longlong_as_double((__double_as_longlong(s) & (0x7ffll << 52)) + (1ll << 52));
                stop = stop || s + (X - before) >= next;
            }
            const unsigned long long m = __ballot(stop && lane >= pos);
            const int first = m ? __ffsll(m) - 1 : HB_WAVE;
            if (first > (int)pos) S = (float)(s + (__shfl(X, first - 1) - before));
            if (first == HB_WAVE) break;
            S = wide_replay16(S, a, first);
            before = __shfl(X, first);
            pos = (uint32_t)first + 1;
        }
    }
    return S;
}

// estimate of a row from its (wave-reduced) sums; every lane returns it
template <int P, class Row>
__device__ __forceinline__ float wide_estimate(const HbDev &d, const WideSum &w, Row row)
{
    if (w.z > 0) {
        const float lc = d.lc[w.z];
        if ((double)lc <= d.lc_thr) return lc;
    }
    float S;
    // k = sum of 2^(mx - M) as at p <= 10: below 2^24 the f32 sum is exact
    if (w.mx <= 24 && (w.s24 >> (24 - w.mx)) < (1ull << 24))
        S = ldexpf((float)(uint32_t)(w.s24 >> (24 - w.mx)), -(int)w.mx);
    else
        S = wide_sequential_sum<Wide<P>::CHUNKS>(w.mx, row);
    float est = (float)((double)d.am / (double)S);
    if (est <= d.five_m) est = (float)((double)est - hb_bias_lookup(d.bias, est));
    return est;
}

// acc[c] = max over the rows of nb[0 .. len), chunks c0 .. c0 + CG - 1.  kChanged: rows of
// the nodes in `bits` only.
template <int P, Gather kGather>
__device__ __forceinline__ void wide_gather(const uint8_t *__restrict__ in, const uint32_t *__restrict__ bits,
                                            const uint32_t *__restrict__ nb, uint32_t len, int c0, HbAcc *acc,
                                            unsigned long long &gathered)
{
    constexpr int CG = Wide<P>::CG, K = CG == 2 ? 4 : 2;  // rows in flight: eight 1 KiB loads
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    const uint64_t at = (uint64_t)c0 * 1024 + lane * 16;
    for (uint32_t j0 = 0; j0 < len; j0 += HB_WAVE) {
        // 64 ids at a time, a lane each; the listed ones of them become wave-uniform in turn
        const uint32_t id = j0 + lane < len ? nb[j0 + lane] : 0u;
        bool use = j0 + lane < len;
        if (kGather == Gather::kChanged) use = use && bit_test(bits, id);
        unsigned long long m = __ballot(use);
        gathered += __popcll(m);
        while (m) {
            uint32_t v[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {  // past the last one: the last again
                v[k] = (uint32_t)__builtin_amdgcn_readlane((int)id, __ffsll(m) - 1);
                if (m & (m - 1)) m &= m - 1;
                else if (k == K - 1) m = 0;
            }
            uint4 r[K][CG];
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
                for (int c = 0; c < CG; ++c) r[k][c] = *(const uint4 *)(in + ((uint64_t)v[k] << P) + at + c * 1024);
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
                for (int c = 0; c < CG; ++c) hb_acc_max(acc[c], r[k][c]);
        }
    }
}

// acc[c] = max over the insertions of nbh[0 .. len) (iteration 1), chunk by chunk in the
// wavefront's 1,024 LDS words
template <int P>
__device__ __forceinline__ void wide_first(uint32_t *lds, const uint32_t *__restrict__ nbh, uint32_t len, int c0,
                                           HbAcc *acc)
{
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1);
    uint32_t idx = ~0u, rank = 0;
    if (len <= HB_WAVE && lane < len) hb_index_rank(nbh[lane], P, &idx, &rank);
#pragma unroll
    for (int c = 0; c < Wide<P>::CG; ++c) {
        for (int k = 0; k < 16; ++k) lds[k * HB_WAVE + lane] = 0u;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (len <= HB_WAVE) {
            if (idx / 1024 == (uint32_t)(c0 + c)) atomicMax(lds + idx % 1024, rank);
        } else {
            for (uint32_t j = lane; j < len; j += HB_WAVE) {
                hb_index_rank(nbh[j], P, &idx, &rank);
                if (idx / 1024 == (uint32_t)(c0 + c)) atomicMax(lds + idx % 1024, rank);
            }
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint4 x = *(const uint4 *)(lds + lane * 16 + 4 * q);
            w[q] = x.x | (x.y << 8) | (x.z << 16) | (x.w << 24);
        }
        hb_acc_max(acc[c], make_uint4(w[0], w[1], w[2], w[3]));
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// the bound of all sketches packed as registers are (HbDev::sat_row), after the init
__global__ __launch_bounds__(kBlock) void k_pack_bound(HbDev d)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= (1u << d.p) / 4) return;
    const uint4 r = *(const uint4 *)(d.sat_max + 4 * i);
    ((uint32_t *)d.sat_row)[i] = r.x | (r.y << 8) | (r.z << 16) | (r.w << 24);
}

template <int P>
__global__ __launch_bounds__(kBlock) void k_init_wide(HbDev d)
{
    constexpr uint32_t M = 1u << P;
    const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t u = (uint32_t)(gtid / HB_WAVE), lane = (uint32_t)(gtid % HB_WAVE);
    if (u >= d.n) return;
    uint32_t idx, rank;
    hb_index_rank(d.node_id ? d.node_id[u] : u, P, &idx, &rank);
    const uint32_t e0 = d.off[u], deg = d.off[u + 1] - e0;
    const bool isolated = deg == 0;
    for (uint32_t c = 0; c < M / 1024; ++c) {
        const uint32_t base = c * 1024 + lane * 16;
        uint32_t w[4] = {0, 0, 0, 0};
        if (idx >= base && idx < base + 16) w[(idx - base) / 4] = rank << (8 * (idx % 4));
        const uint4 r = make_uint4(w[0], w[1], w[2], w[3]);
        *(uint4 *)(d.regs0 + ((uint64_t)u << P) + base) = r;
        if (isolated) *(uint4 *)(d.regs1 + ((uint64_t)u << P) + base) = r;
    }
    if (lane == 0) {
        d.est[u] = d.lc[M - 1];  // one non-zero register: linear counting with m-1 zeros
        d.dist[u] = 0.0;
        d.inv[u] = 0.0;
        if (d.sat_max) {  // as k_init
            const uint32_t w = d.sat_sym && deg == 1 ? d.nbr[e0] : 0u;
            const bool alone = d.sat_sym && (deg == 0 || (deg == 1 && d.off[w + 1] - d.off[w] == 1));
            if (!alone && d.sat_max[idx] < rank) atomicMax(d.sat_max + idx, rank);
        }
    }
}

// kNodes: the listed nodes; kHubs: hub nodes, whose rows come from the partial rows of their
// tasks (list: the hubs, then each one's first task, then its number of tasks)
enum class WideKind { kNodes, kHubs };

template <int P, bool kFirst, WideKind kKind>
__global__ __launch_bounds__(kBlock) void k_union_wide(HbDev d, const uint32_t *__restrict__ list,
                                                       const uint32_t *__restrict__ htask0,
                                                       const uint32_t *__restrict__ hntask, uint32_t count,
                                                       int slot_id)
{
    using W = Wide<P>;
    const HbIterState *st = d.st;
    if (st->done) return;
    constexpr bool kHash = kFirst && kKind == WideKind::kNodes;
    __shared__ __attribute__((aligned(16))) uint32_t s_first[kHash ? kBlock * 16 : 4];
    const uint32_t it = st->iter;
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1), w = threadIdx.x / HB_WAVE;
    uint32_t *lds = s_first + (kHash ? w * 1024 : 0);
    HbView v{};
    v.off = d.off;
    v.in = st->parity ? d.regs1 : d.regs0;
    v.out = st->parity ? d.regs0 : d.regs1;
    v.dist = d.dist;
    v.inv = d.inv;
    v.bitsR = (it & 1u) ? d.bits0 : d.bits1;
    v.bitsW = (it & 1u) ? d.bits1 : d.bits0;
    v.t = st->t;
    v.inv_t = st->inv_t;
    v.use_frontier = d.frontier && it > 1 && !st->skip_scan;
    v.sym = d.sat_sym != 0;
    if (d.sat_max && !kFirst) {
        v.satR = hb_saturated(d, it - 1);
        v.satW = hb_saturated(d, it);
        v.sat_scan = st->sat_scan != 0;
    }
    HbCounts cn;
    unsigned long long c_gathered = 0;

    for (uint32_t i = blockIdx.x * (kBlock / HB_WAVE) + w; i < count; i += gridDim.x * (kBlock / HB_WAVE)) {
        const uint32_t u = __builtin_amdgcn_readfirstlane(list[i]);
        const uint32_t e0 = d.off[u], deg = d.off[u + 1] - e0;
        const uint32_t *__restrict__ nb = d.nbr + e0;
        const uint8_t *own_row = v.in + ((uint64_t)u << P) + lane * 16;
        uint8_t *out_row = v.out + ((uint64_t)u << P) + lane * 16;
        const uint8_t *bound = d.sat_row + lane * 16;
        const uint32_t t0 = kKind == WideKind::kHubs ? htask0[i] : 0u, nt = kKind == WideKind::kHubs ? hntask[i] : 0u;
        if (v.satR && bit_test(v.satR, u)) {  // nothing can change; keep both buffers complete
            if (bit_test(v.bitsR, u))
                for (int c = 0; c < W::CHUNKS; ++c) *(uint4 *)(out_row + c * 1024) = *(const uint4 *)(bound + c * 1024);
            continue;
        }
        bool sat = false;
        uint32_t scanned = deg;
        if constexpr (kKind == WideKind::kNodes) {
            if (v.sat_scan) {
                uint32_t k = 0;
                sat = sat_neighbour<HB_WAVE>(v.satR, nb, deg, lane, k);
                if (sat) scanned = k;
            }
        }
        bool active = true;
        if (kKind == WideKind::kHubs) {
            uint32_t any = 0;
            for (uint32_t j = lane; j < nt; j += HB_WAVE) any |= d.chunk_flag[t0 + j];
            active = hb_copy_or<HB_WAVE>(any) != 0;
        } else if (v.use_frontier && !sat) {
            uint32_t any = 0;
            for (uint32_t j = lane; j < deg; j += HB_WAVE) any |= bit_test(v.bitsR, nb[j]);
            active = hb_copy_or<HB_WAVE>(any) != 0;
        }
        if (!active) {
            if (bit_test(v.bitsR, u))
                for (int c = 0; c < W::CHUNKS; ++c) *(uint4 *)(out_row + c * 1024) = *(const uint4 *)(own_row + c * 1024);
            continue;
        }
        WideSum sum;
        uint32_t diffw = 0;  // bit 0: a register rose; bit 1: one is below the bound
        uint4 row[W::CG];    // the last pass's chunks: all of the row up to p = 12
        for (int c0 = 0; c0 < W::CHUNKS; c0 += W::CG) {
            if (sat) {
#pragma unroll
                for (int c = 0; c < W::CG; ++c) row[c] = *(const uint4 *)(bound + (c0 + c) * 1024);
                diffw = 1u;
            } else {
                HbAcc acc[W::CG];
                uint4 own[W::CG];
#pragma unroll
                for (int c = 0; c < W::CG; ++c) {
                    own[c] = *(const uint4 *)(own_row + (c0 + c) * 1024);
                    acc[c] = hb_acc(own[c]);
                }
                unsigned long long g = 0;
                if constexpr (kKind == WideKind::kHubs) {
                    for (uint32_t j = 0; j < nt; ++j)
                        if (d.chunk_flag[t0 + j])
#pragma unroll
                            for (int c = 0; c < W::CG; ++c)
                                hb_acc_max(acc[c], *(const uint4 *)(d.scratch + ((uint64_t)(t0 + j) << P) +
                                                                    (c0 + c) * 1024 + lane * 16));
                } else if constexpr (kFirst) {
                    wide_first<P>(lds, d.orig + e0, deg, c0, acc);
                } else if (v.use_frontier) {
                    wide_gather<P, Gather::kChanged>(v.in, v.bitsR, nb, deg, c0, acc, g);
                } else {
                    wide_gather<P, Gather::kAll>(v.in, nullptr, nb, deg, c0, acc, g);
                }
                if (c0 == 0) c_gathered += g;
#pragma unroll
                for (int c = 0; c < W::CG; ++c) {
                    row[c] = hb_acc_get(acc[c]);
                    diffw |= (row[c].x != own[c].x) | (row[c].y != own[c].y) | (row[c].z != own[c].z) |
                             (row[c].w != own[c].w);
                    if (v.satR) {
                        const uint4 f = *(const uint4 *)(bound + (c0 + c) * 1024);
                        diffw |= ((row[c].x != f.x) | (row[c].y != f.y) | (row[c].z != f.z) | (row[c].w != f.w)) << 1;
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < W::CG; ++c) {
                *(uint4 *)(out_row + (c0 + c) * 1024) = row[c];
                sum.add(row[c]);
            }
        }
        sum.reduce();
        diffw = hb_copy_or<HB_WAVE>(diffw);
        const float curr = wide_estimate<P>(d, sum, [&](int c) {
            if constexpr (W::PASSES == 1) {
                uint4 x = row[0];
#pragma unroll
                for (int k = 1; k < W::CG; ++k)
                    if (c == k) x = row[k];
                return x;
            } else {
                return *(const uint4 *)(out_row + c * 1024);  // this lane's own stores
            }
        });
        if (lane == 0) {
            const float prev = d.est[u];
            if (accumulate(v, u, prev, curr)) cn.inc += 1;
            d.est[u] = curr;
            if (diffw & 1u) {
                atomicOr(v.bitsW + (u >> 5), 1u << (u & 31u));
                cn.chg += 1;
            }
            if (v.satR && !(diffw & 2u) && sat_allowed(v, nb, deg)) {
                bit_set(v.satW, u);
                cn.sat += deg;
            }
            if (kKind == WideKind::kNodes) cn.arcs += scanned;
            cn.nodes += 1;
        }
    }
    block_add(cn.inc, cn.arcs, cn.nodes, cn.chg, lane == 0 ? c_gathered : 0, cn.sat, d, slot_id);
}

// one task of a hub's list: a wavefront per pass of its partial row
template <int P, bool kFirst>
__global__ __launch_bounds__(kBlock) void k_chunk_wide(HbDev d, const uint32_t *__restrict__ tnode,
                                                       const uint32_t *__restrict__ tbeg,
                                                       const uint32_t *__restrict__ tend, uint32_t ntasks)
{
    using W = Wide<P>;
    const HbIterState *st = d.st;
    if (st->done) return;
    __shared__ __attribute__((aligned(16))) uint32_t s_first[kFirst ? kBlock * 16 : 4];
    const uint32_t it = st->iter;
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1), w = threadIdx.x / HB_WAVE;
    const uint8_t *__restrict__ in = st->parity ? d.regs1 : d.regs0;
    const uint32_t *__restrict__ bitsR = (it & 1u) ? d.bits0 : d.bits1;
    const bool use_frontier = d.frontier && it > 1 && !st->skip_scan;
    const uint32_t *satR = d.sat_max && !kFirst ? hb_saturated(d, it - 1) : nullptr;
    const bool sat_scan = satR && st->sat_scan;
    unsigned long long c_arcs = 0, c_gathered = 0;
    for (uint32_t i = blockIdx.x * (kBlock / HB_WAVE) + w; i < ntasks * W::PASSES; i += gridDim.x * (kBlock / HB_WAVE)) {
        const uint32_t task = __builtin_amdgcn_readfirstlane(i / W::PASSES);
        const int c0 = (int)(i % W::PASSES) * W::CG;
        const uint32_t eb = tbeg[task], len = tend[task] - eb;
        const uint32_t *__restrict__ nb = d.nbr + eb;
        bool active = !(satR && bit_test(satR, tnode[task]));
        uint32_t scanned = len;
        const bool sat = active && sat_scan && sat_neighbour<HB_WAVE>(satR, nb, len, lane, scanned);
        if (active && use_frontier && !sat) {
            uint32_t any = 0;
            for (uint32_t j = lane; j < len; j += HB_WAVE) any |= bit_test(bitsR, nb[j]);
            active = hb_copy_or<HB_WAVE>(any) != 0;
        }
        if (lane == 0 && c0 == 0) d.chunk_flag[task] = active ? 1u : 0u;
        if (!active) continue;
        uint8_t *out = d.scratch + ((uint64_t)task << P) + c0 * 1024 + lane * 16;
        if (c0 == 0) c_arcs += sat ? scanned : len;
        if (sat) {  // the hub becomes the bound through this task
#pragma unroll
            for (int c = 0; c < W::CG; ++c)
                *(uint4 *)(out + c * 1024) = *(const uint4 *)(d.sat_row + (c0 + c) * 1024 + lane * 16);
            continue;
        }
        HbAcc acc[W::CG];
#pragma unroll
        for (int c = 0; c < W::CG; ++c) acc[c] = hb_acc(make_uint4(0, 0, 0, 0));
        unsigned long long g = 0;
        if constexpr (kFirst) wide_first<P>(s_first + w * 1024, d.orig + eb, len, c0, acc);
        else if (use_frontier) wide_gather<P, Gather::kChanged>(in, bitsR, nb, len, c0, acc, g);
        else wide_gather<P, Gather::kAll>(in, nullptr, nb, len, c0, acc, g);
        if (c0 == 0) c_gathered += g;
#pragma unroll
        for (int c = 0; c < W::CG; ++c) *(uint4 *)(out + c * 1024) = hb_acc_get(acc[c]);
    }
    block_add(0, lane == 0 ? c_arcs : 0, 0, 0, lane == 0 ? c_gathered : 0, 0, d, HB_SLOT_CHUNK);
}

template <int P>
__global__ __launch_bounds__(kBlock) void k_estimates_wide(HbDev d, const uint8_t *__restrict__ regs,
                                                           float *__restrict__ out)
{
    const uint32_t lane = threadIdx.x & (HB_WAVE - 1), w = threadIdx.x / HB_WAVE;
    for (uint32_t u = blockIdx.x * (kBlock / HB_WAVE) + w; u < d.n; u += gridDim.x * (kBlock / HB_WAVE)) {
        const uint8_t *row = regs + ((uint64_t)u << P) + lane * 16;
        WideSum sum;
#pragma unroll 4
        for (int c = 0; c < Wide<P>::CHUNKS; ++c) sum.add(*(const uint4 *)(row + c * 1024));
        sum.reduce();
        const float e = wide_estimate<P>(d, sum, [&](int c) { return *(const uint4 *)(row + c * 1024); });
        if (lane == 0) out[u] = e;
    }
}

// ---------------------------------------------------------------------------
// neighbourhood function N(t) = sum_u est_t(u), summed exactly in 128-bit fixed
// point with 40 fractional bits (every estimate is >= 1, whose f32 ulp >= 2^-23)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_nf(HbDev d)
{
    const HbIterState *st = d.st;
    if (st->done) return;
    unsigned long long lo = 0, hi = 0;
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < d.n; u += gridDim.x * blockDim.x) {
        const uint32_t b = __float_as_uint(d.est[u]);
        const int e = (int)((b >> 23) & 0xffu);
        const unsigned long long mant = (e ? (1ull << 23) : 0ull) | (b & 0x7fffffu);
        const int sh = (e ? e : 1) - 127 - 23 + 40;  // value * 2^40 = mant * 2^sh
        unsigned long long vlo, vhi;
        if (sh >= 64) { vlo = 0; vhi = mant << (sh - 64); }
        else if (sh > 0) { vlo = mant << sh; vhi = sh > 40 ? (mant >> (64 - sh)) : 0ull; }
        else { vlo = mant >> (-sh); vhi = 0; }
        const unsigned long long nlo = lo + vlo;
        hi += vhi + (nlo < lo);
        lo = nlo;
    }
    // wave reduction with carries
#pragma unroll
    for (int s = 1; s < HB_WAVE; s <<= 1) {
        const unsigned long long olo = __shfl_xor(lo, s), ohi = __shfl_xor(hi, s);
        const unsigned long long nlo = lo + olo;
        hi = hi + ohi + (nlo < lo);
        lo = nlo;
    }
    if ((threadIdx.x & (HB_WAVE - 1)) == 0) {
        HbIterRec *r = d.rec;
        const unsigned long long old = atomicAdd(&r->nf_lo, lo);
        atomicAdd(&r->nf_hi, hi + ((old + lo) < old ? 1ull : 0ull));
    }
}

// estimates after iteration t <= snap_k (surrogate inputs)
__global__ __launch_bounds__(kBlock) void k_snapshot(HbDev d)
{
    const HbIterState *st = d.st;
    if (st->done || st->iter > d.snap_k) return;
    float *dst = d.snaps + (uint64_t)(st->iter - 1) * d.n;
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < d.n; u += gridDim.x * blockDim.x) dst[u] = d.est[u];
}

// end of iteration t: the counter copies summed into the host's ring record and cleared, the
// termination rule (hyper_ball.rs:833-849) and the buffer swap; one wavefront
__global__ __launch_bounds__(HB_WAVE) void k_finalize(HbDev d)
{
    HbIterState *st = d.st;
    if (st->done) return;
    const uint32_t it = st->iter, lane = threadIdx.x;
    HbIterRec &rec = d.host_rec[it % HB_REC_RING];
    constexpr uint32_t kCounts = 5 * HB_NSLOT + 1;
    static_assert(kCounts <= HB_COUNT_STRIDE && HB_COUNT_STRIDE <= HB_WAVE / 2, "a lane per counter, two copies at a time");
    const uint32_t at = lane % HB_COUNT_STRIDE;
    unsigned long long t = 0;
#pragma unroll
    for (uint32_t k = lane / HB_COUNT_STRIDE; k < HB_COUNT_COPIES; k += HB_WAVE / HB_COUNT_STRIDE) {
        unsigned long long *p = d.counts + k * HB_COUNT_STRIDE + at;
        t += *p;
        *p = 0ull;
    }
#pragma unroll
    for (uint32_t o = HB_COUNT_STRIDE; o < HB_WAVE; o <<= 1) t += __shfl_xor(t, o);
    if (lane < kCounts) {  // inc, arcs, nodes, chg, gathered per slot, then sat: as in HbIterRec
        unsigned long long *p = lane < 5 * HB_NSLOT ? &rec.inc[0] + lane : &rec.sat;
        *p = t;
    }
    auto slots = [&](uint32_t kind) {
        unsigned long long x = 0;
        for (uint32_t k = 0; k < HB_NSLOT; ++k) x += __shfl(t, kind * HB_NSLOT + k);
        return x;
    };
    const unsigned long long inc = slots(0), chg = slots(3), sat = __shfl(t, 5 * HB_NSLOT);
    if (lane != 0) return;
    const bool stop = inc == 0 || (st->max_iters && it >= st->max_iters);
    rec.nf_lo = d.rec->nf_lo;
    rec.nf_hi = d.rec->nf_hi;
    rec.push = d.rec->push;
    rec.iter = it;
    rec.done = stop ? 1u : 0u;
    rec.converged = inc == 0 ? 1u : 0u;
    if (stop) {
        st->done = 1;
        st->executed = it;
        st->converged = inc == 0;
        return;
    }
    st->iter = it + 1;
    st->parity ^= 1u;
    // Iteration 1 marks no node saturated.  Iteration 2 recomputes every node, so that from then
    // on a node whose sketch is the bound is marked, and one that a saturated neighbour raises
    // has changed.  (Almost every node changes in iteration 1 anyway.)
    const bool mark = it == 1 && d.sat_max;
    st->skip_scan = mark || 2 * chg > (unsigned long long)d.n_linked;
    // push when few nodes changed (on R-MAT-24 a push pass at 24% changed nodes whose lists
    // hold 2% of the arcs measured slower than the scan with selective gathers)
    st->push = !mark && d.sym && d.p <= 10 && d.frontier && 16 * chg <= (unsigned long long)d.n_linked;
    // a search that finds nothing costs a node about a quarter of its gather on short lists
    // (Erdos-Renyi, n = 65,536, degree 32: 74 against 60 us an iteration), one that finds a
    // neighbour saves all of it: search once a node has one in eight such neighbours on average
    st->sat_arcs += sat;
    st->sat_scan = 8 * st->sat_arcs >= (unsigned long long)d.n_linked;
    st->t = st->t + 1.0;
    st->inv_t = __ddiv_rn(1.0, st->t);
}

// ---------------------------------------------------------------------------
// epilogues
// ---------------------------------------------------------------------------
template <int P>
__global__ __launch_bounds__(kBlock) void k_estimates(HbDev d, const uint8_t *__restrict__ regs,
                                                      float *__restrict__ out)
{
    constexpr uint32_t M = 1u << P, G = M / 16;
    HB_TABLES_LDS(P, d, tb)
    const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t u = (uint32_t)(gtid / G), cl = (uint32_t)(gtid % G);
    if (u >= d.n) return;
    const uint4 r = *(const uint4 *)(regs + ((uint64_t)u << P) + cl * 16);
    const float e = hb_estimate_copy<G>(tb, r);
    if (cl == 0) out[u] = e;
}

// hyper_ball.rs:434-555: closeness (:447-466), harmonic (:500-518, guard on dist),
// Lin (:540-547, 1 when dist is not normal)
__global__ __launch_bounds__(kBlock) void k_centrality(HbDev d, const float *__restrict__ est,
                                                       int kind, int normalize, double *__restrict__ out)
{
    const double nf = (double)d.n - 1.0;
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < d.n; u += gridDim.x * blockDim.x) {
        const double dd = d.dist[u];
        const double e = (double)est[u];
        const bool normal = isnormal(dd);
        double r;
        if (kind == 0) r = !normal ? 0.0 : (normalize ? __ddiv_rn(__dsub_rn(e, 1.0), dd) : __ddiv_rn(nf, dd));
        else if (kind == 1) r = !normal ? 0.0 : (normalize ? __ddiv_rn(d.inv[u], __dsub_rn(e, 1.0)) : __ddiv_rn(d.inv[u], nf));
        else {
            const double x = __dsub_rn(e, 1.0);
            r = !normal ? 1.0 : __ddiv_rn(__dmul_rn(x, x), dd);
        }
        out[u] = r;
    }
}

// ---------------------------------------------------------------------------
// host-side launchers
// ---------------------------------------------------------------------------
static unsigned grid_for(uint64_t threads, unsigned cap)
{
    const uint64_t b = (threads + kBlock - 1) / kBlock;
    return (unsigned)(b < 1 ? 1 : (b > cap ? cap : b));
}

template <int P, bool kFirst>
static hipError_t launch_union_T(const HbDev &d, const uint32_t *list, uint32_t base, uint32_t count, int T,
                                 unsigned max_blocks, int slot, hipStream_t s)
{
    constexpr int G = (1 << P) / 16;
    const unsigned grid = grid_for((uint64_t)count * T, max_blocks);
    switch (T) {
#define HB_CASE(TT)                                                                        \
    case TT:                                                                               \
        if constexpr (TT >= G) {                                                           \
            k_union<P, TT, kFirst><<<grid, kBlock, 0, s>>>(d, list, base, count, slot);            \
            return hipGetLastError();                                                      \
        }                                                                                  \
        break;
        HB_CASE(1) HB_CASE(2) HB_CASE(4) HB_CASE(8) HB_CASE(16) HB_CASE(32) HB_CASE(64)
#undef HB_CASE
    }
    return hipErrorInvalidValue;
}

#define HB_DISPATCH_P(p, ...)                              \
    switch (p) {                                           \
    case 4: { constexpr int P = 4; __VA_ARGS__; } break;   \
    case 5: { constexpr int P = 5; __VA_ARGS__; } break;   \
    case 6: { constexpr int P = 6; __VA_ARGS__; } break;   \
    case 7: { constexpr int P = 7; __VA_ARGS__; } break;   \
    case 8: { constexpr int P = 8; __VA_ARGS__; } break;   \
    case 9: { constexpr int P = 9; __VA_ARGS__; } break;   \
    case 10: { constexpr int P = 10; __VA_ARGS__; } break; \
    default: return hipErrorInvalidValue;                  \
    }

#define HB_DISPATCH_WIDE(p, ...)                            \
    switch (p) {                                            \
    case 11: { constexpr int P = 11; __VA_ARGS__; } break;  \
    case 12: { constexpr int P = 12; __VA_ARGS__; } break;  \
    case 13: { constexpr int P = 13; __VA_ARGS__; } break;  \
    case 14: { constexpr int P = 14; __VA_ARGS__; } break;  \
    case 15: { constexpr int P = 15; __VA_ARGS__; } break;  \
    case 16: { constexpr int P = 16; __VA_ARGS__; } break;  \
    default: return hipErrorInvalidValue;                   \
    }

hipError_t launch_init(const HbDev &d, hipStream_t s)
{
    if (d.p > 10) {
        HB_DISPATCH_WIDE(d.p, {
            k_init_wide<P><<<(unsigned)(((uint64_t)d.n * HB_WAVE + kBlock - 1) / kBlock), kBlock, 0, s>>>(d);
        });
        if (d.sat_max) k_pack_bound<<<((1u << d.p) / 4 + kBlock - 1) / kBlock, kBlock, 0, s>>>(d);
        return hipGetLastError();
    }
    // k_init stores the linear-counting estimate of m - 1 zeros for every node; it is what
    // the estimator returns for a one-insertion sketch when LC <= the HLL++ threshold,
    // which holds at every p (LC < 1.04, thresholds >= 10), checked here with the same
    // expression the LC table is filled with
    const double m = (double)(1u << d.p);
    if ((double)(float)(m * std::log(m / (m - 1.0))) > d.lc_thr) return hipErrorInvalidValue;
    HB_DISPATCH_P(d.p, {
        k_init<P><<<(unsigned)(((uint64_t)d.n + kBlock - 1) / kBlock), kBlock, 0, s>>>(d);
    });
    return hipGetLastError();
}

hipError_t launch_fill(uint32_t *p, uint64_t count, uint32_t value, hipStream_t s)
{
    if (count == 0) return hipSuccess;
    k_fill_u32<<<grid_for(count, 4096), kBlock, 0, s>>>(p, count, value);
    return hipGetLastError();
}

hipError_t launch_start(HbIterState *st, const HbIterState &st0, uint32_t *p, uint64_t count, hipStream_t s)
{
    k_start<<<grid_for(count, 4096), kBlock, 0, s>>>(st, st0, p, count);
    return hipGetLastError();
}

hipError_t launch_iteration(const HbDev &d, const HbSchedule &sc, bool first, bool nf, hipStream_t s,
                            hipEvent_t *ev)
{
    const uint32_t words = (d.n + 31) / 32;
    const bool push_possible = d.sym && d.p <= 10 && d.frontier;
    // where push iterations can occur k_begin also marks, one wavefront per bitmap word
    k_begin<<<push_possible ? grid_for((uint64_t)words * HB_WAVE, 8192) : grid_for(words, 2048), kBlock, 0, s>>>(
        d, words);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (push_possible && !first) {  // returns at once unless this is a push iteration
        HB_DISPATCH_P(d.p, k_push_compact<P><<<grid_for(words, 4096), kBlock, 0, s>>>(d, words));
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    for (int b = 0; b < sc.nbins; ++b) {
        if (sc.bin_count[b] == 0) continue;
        if (ev) (void)hipEventRecord(ev[2 * b], s);
        if (d.p > 10) {
            HB_DISPATCH_WIDE(d.p, {
                auto *nodes = first ? k_union_wide<P, true, WideKind::kNodes> : k_union_wide<P, false, WideKind::kNodes>;
                nodes<<<grid_for((uint64_t)sc.bin_count[b] * HB_WAVE, sc.max_blocks), kBlock, 0, s>>>(
                    d, sc.bin_list[b], nullptr, nullptr, sc.bin_count[b], b);
                e = hipGetLastError();
            });
        } else {
            // k_union_rows and k_union each return at once in the iterations the other runs
            if (rows_bin(d, sc, b)) {
                const unsigned grid = grid_for(sc.bin_count[b], sc.max_blocks);
                if (d.p == 5) k_union_rows<5><<<grid, kBlock, 0, s>>>(d, sc.bin_base[b], sc.bin_count[b], b);
                else k_union_rows<6><<<grid, kBlock, 0, s>>>(d, sc.bin_base[b], sc.bin_count[b], b);
                e = hipGetLastError();
                if (e != hipSuccess) return e;
            }
            if (!(first && rows_bin(d, sc, b)))
                HB_DISPATCH_P(d.p, {
                    auto *launch = first ? launch_union_T<P, true> : launch_union_T<P, false>;
                    e = launch(d, sc.bin_list[b], sc.bin_base[b], sc.bin_count[b], sc.bin_team[b], sc.max_blocks, b, s);
                });
        }
        if (ev) (void)hipEventRecord(ev[2 * b + 1], s);
        if (e != hipSuccess) return e;
    }
    if (sc.ntasks && d.p > 10) {
        HB_DISPATCH_WIDE(d.p, {
            auto *chunk = first ? k_chunk_wide<P, true> : k_chunk_wide<P, false>;
            auto *hubs = first ? k_union_wide<P, true, WideKind::kHubs> : k_union_wide<P, false, WideKind::kHubs>;
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_CHUNK], s);
            chunk<<<grid_for((uint64_t)sc.ntasks * Wide<P>::PASSES * HB_WAVE, sc.max_blocks), kBlock, 0, s>>>(
                d, sc.task_node, sc.task_beg, sc.task_end, sc.ntasks);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_CHUNK + 1], s);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_MERGE], s);
            hubs<<<grid_for((uint64_t)sc.nhubs * HB_WAVE, sc.max_blocks), kBlock, 0, s>>>(
                d, sc.hub_node, sc.hub_task0, sc.hub_ntask, sc.nhubs, HB_SLOT_MERGE);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_MERGE + 1], s);
        });
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    } else if (sc.ntasks) {
        HB_DISPATCH_P(d.p, {
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_CHUNK], s);
            auto *chunk = first ? k_chunk<P, true> : k_chunk<P, false>;
            chunk<<<grid_for((uint64_t)sc.ntasks * HB_WAVE, sc.max_blocks), kBlock, 0, s>>>(
                d, sc.task_node, sc.task_beg, sc.task_end, sc.ntasks);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_CHUNK + 1], s);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_MERGE], s);
            k_merge<P><<<grid_for((uint64_t)sc.nhubs * HB_WAVE, sc.max_blocks), kBlock, 0, s>>>(
                d, sc.hub_node, sc.hub_task0, sc.hub_ntask, sc.nhubs);
            if (ev) (void)hipEventRecord(ev[2 * HB_SLOT_MERGE + 1], s);
        });
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (nf) {
        k_nf<<<grid_for(d.n, 1024), kBlock, 0, s>>>(d);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (d.snap_k) {
        k_snapshot<<<grid_for(d.n, 4096), kBlock, 0, s>>>(d);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    k_finalize<<<1, HB_WAVE, 0, s>>>(d);
    return hipGetLastError();
}

hipError_t arc_fingerprints(const uint32_t *off, const uint32_t *nbr, uint32_t n, uint64_t arcs,
                            unsigned long long *work, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    // no more blocks than there are arcs for their lanes: a small graph's search and sum
    // take 7 us instead of 37
    const uint64_t want = (arcs + (uint64_t)kBlock * kFpArcs - 1) / ((uint64_t)kBlock * kFpArcs);
    const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(want, kFingerprintBlocks));
    k_arc_fingerprint<<<blocks, kBlock, 0, s>>>(off, nbr, n, arcs, work + 4);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return sum_columns(work + 4, blocks, 4, work, s);
}

// out[k] = sum over r < rows of part[r * cols + k], one block per column, a fixed
// summation order (so f64 sums are reproducible)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sum_columns(const T *part, uint32_t rows, uint32_t cols, T *out)
{
    __shared__ T red[kBlock];
    const uint32_t k = blockIdx.x;
    T t = 0;
    for (uint32_t r = threadIdx.x; r < rows; r += kBlock) t += part[(uint64_t)r * cols + k];
    red[threadIdx.x] = t;
    __syncthreads();
    for (uint32_t w = kBlock / 2; w; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = red[0];
}

template <typename T>
hipError_t sum_columns(const T *part, uint32_t rows, uint32_t cols, T *out, hipStream_t s)
{
    if (cols == 0) return hipSuccess;
    k_sum_columns<T><<<cols, kBlock, 0, s>>>(part, rows, cols, out);
    return hipGetLastError();
}
template hipError_t sum_columns<unsigned long long>(const unsigned long long *, uint32_t, uint32_t,
                                                    unsigned long long *, hipStream_t);
template hipError_t sum_columns<double>(const double *, uint32_t, uint32_t, double *, hipStream_t);

hipError_t launch_estimates(const HbDev &d, const uint8_t *regs, float *out, hipStream_t s)
{
    if (d.p > 10) {
        HB_DISPATCH_WIDE(d.p, {
            k_estimates_wide<P><<<grid_for((uint64_t)d.n * HB_WAVE, 8192), kBlock, 0, s>>>(d, regs, out);
        });
        return hipGetLastError();
    }
    HB_DISPATCH_P(d.p, {
        const uint64_t threads = (uint64_t)d.n * ((1 << P) / 16);
        k_estimates<P><<<(unsigned)((threads + kBlock - 1) / kBlock), kBlock, 0, s>>>(d, regs, out);
    });
    return hipGetLastError();
}

hipError_t launch_centrality(const HbDev &d, const float *est, int kind, int normalize, double *out,
                             hipStream_t s)
{
    k_centrality<<<grid_for(d.n, 4096), kBlock, 0, s>>>(d, est, kind, normalize, out);
    return hipGetLastError();
}

}  // namespace hb
