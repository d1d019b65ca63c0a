// hb_exact.hip -- exact BFS centralities on the GPU: up to 2,048 breadth-first searches at
// once in a slice (one bit lane per source, SW u64 words per node), several slices side
// by side, advanced one level per set of launches.
//
// Semantics follow the reference's BFS (src/trails/bfs.rs:199-234): the source is
// queued with distance 0 but not marked visited, so it is rediscovered one step
// after the first node with an arc back to it (distance 1 through a self-loop) and
// counted like any other node.  Level-synchronous form, per source bit:
//     visited = {}, frontier = {source}
//     level d: next = nodes with an arc from a frontier node;  newly = next \ visited
//              visited |= newly, frontier = newly, reachable += |newly|, total += d |newly|
// which discovers exactly the nodes (and distances) of the reference's FIFO queue.
//
// Level 1 pushes the sources' own arcs (k_bfs_sources).  Later levels pull: a node
// that some live source has not reached ORs the frontier rows of the nodes with an arc to
// it (its list on a symmetric CSR; otherwise the reversed CSR, built once per call).  No
// atomics, and a row of 2,048 searches costs two cache lines where a single 8-byte word takes
// one: the pull is bound by the rate of random requests, not by bytes, so the searches of a
// slice share them.  2,048 sources of R-MAT-20 (31.4M arcs): 4.6 ms of pulls over 7 levels (64
// sources at a time: 22 ms of pulls and 9 of per-pass bookkeeping); all 16,384 sources of a de
// Bruijn graph (131,068 arcs): 0.8 ms for the call instead of 64.
// What keeps a level cheap when little is left to do:
//   - a byte per node says whether its frontier row holds any bit; rows without are neither
//     written nor read, and an arc costs its id and that byte;
//   - a source whose last level found nothing leaves the live mask, so that nodes it cannot
//     reach do not look for it again;
//   - a list is left as soon as every wanted bit has appeared;
//   - with few sources (rows of two words) a level whose frontier has few arcs pushes them
//     (k_bfs_push): a node in a component without a source wants bits for ever, and a pull scans
//     its list in every level.  A path of 2,000 nodes beside R-MAT-18, 64 sources on the path: 45 ms,
//     245 when every level pulled; a grid of 1,000 x 1,000, 1 source: 54 and 67 ms.
//
// Per-source sums, bit-identical to the reference's:
//   reachable : integer count (BFSDists::recheable)
//   total     : Σ d as an integer; the reference's f64 running sum of integers is
//               exact while it stays below 2^53 (16.7M nodes at distance 1000 is 2^34)
//   inv_sum   : Σ_v 1/d(v) over v = 0..n-1 in node order, 1/d a correctly rounded
//               f64 division and 0 for unreached nodes (exact.rs:386-396: an iterator
//               sum over get_distances()).  The order fixes the rounding; see k_bfs_harmonic
//               for how all but a few of the adds are done in any order all the same.
#include <hip/hip_runtime.h>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "../../include/sparkx_hb.h"
#include "hb_kernels.h"

namespace hb {

constexpr int kBfsBlock = 256;
constexpr uint32_t kBfsChunk = 128;    // nodes per count: at most 128 fits a byte
constexpr uint32_t kBfsHubDeg = 256;   // longer lists are cut into kBfsHubArcs-arc tasks
constexpr uint32_t kBfsHubArcs = 1024;
constexpr uint32_t kBfsPlanes = 4;     // bits of a kept distance
constexpr uint32_t kBfsKeep = (1u << kBfsPlanes) - 1;  // levels whose distances can be kept
// A level of rows of two words pushes when the arcs out of its frontier are at most an eighth of
// all arcs (a sixteenth: 64 sources of R-MAT-20 take 7% longer, paths and grids the same), on graphs
// of at least kBfsPushArcs: below, a pull scans all arcs in about the time of the push's launch.
// Wider rows always pull, as that one scan serves all their sources (256 sources on a path
// beside R-MAT-18: 225 ms; 267 when passes of 64 pushed).
constexpr uint32_t kBfsPush = 8;
constexpr uint64_t kBfsPushArcs = 1ull << 20;
// Directed graphs: up to this many sources (one row of two words) every level pushes and the arcs
// are not reversed, which would take memory for 5 words an arc and, on R-MAT-20 with 8.4M arcs, most
// of a call (1 / 64 / 128 sources: 0.97 / 1.45 / 1.86 ms, 2.66 / 2.78 / 2.76 when they were).  From
// 129 on the wider rows' pulls pay for it: 129 and 256 sources 2.9 ms, 2.8 and 4.9 in passes of 64.
constexpr uint32_t kBfsFew = 128;

typedef unsigned long long u64;

// One group of slices, all [slice]-major; a slice covers 64 SW consecutive sources from
// src0 + 64 SW slice.
struct BfsDev {
    const uint32_t *off, *nbr;    // arcs as staged (level 1)
    const uint32_t *ioff, *inbr;  // for each node the tails of the arcs to it
    uint32_t n, src0, src_end;
    uint32_t npad;                // flags per slice: n rounded up to whole chunks
    u64 *visited;                 // [n][SW]
    u64 *live;                    // [SW]: sources still searching
    uint32_t *found;              // [64 SW]: nodes found in the level, zero between levels
    u64 *reach, *total;           // [64 SW]
    uint32_t *done, *levels;      // per slice: nothing found any more; last level that found something
    const uint32_t *hub_node, *hub_first;  // hubs and their tasks (hub h: hub_first[h] ..)
    const uint32_t *task_node, *task_beg, *task_end;
    uint32_t hubs, tasks;
    u64 *part;                    // [tasks][SW]
    // SW == 2: a level may push
    u64 push_arcs;                // if its frontier has at most this many arcs out
    u64 *front;                   // per slice: a bound of them, zero between levels
    uint32_t *push;               // per slice: the next level pushes
    // distances kept for the harmonic sums (null: not), bit-sliced as the rows are: plane k,
    // at k plane_stride, holds bit k of every distance; valid where visited is set
    u64 *plane;
    size_t plane_stride;
};

// The frontier after one level: rows [n][SW] (a row is only valid where its flag is set),
// flags [npad], and the newly found nodes per source counted over kBfsChunk nodes at a time,
// counts [chunks][64 SW] (valid where any is set), any [chunks].
struct BfsLevel {
    u64 *rows;
    uint8_t *flag;
    uint8_t *count;
    uint8_t *any;
};

// The forms a level's launches hold.  kEither: both, and BfsDev::push says which one works.
enum class BfsDir { kPull, kEither, kPush };

template <int SW>
__device__ __forceinline__ bool bfs_pushes(const BfsDev &b, uint32_t slice, BfsDir dir)
{
    return SW == 2 && (dir == BfsDir::kPush || (dir == BfsDir::kEither && b.push[slice]));
}

__device__ __forceinline__ uint32_t bfs_chunks(uint32_t n) { return (n + kBfsChunk - 1) / kBfsChunk; }

template <typename T>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_zero(T *p, uint64_t count)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = T{};
}

// live masks of the sources each slice holds; per-source sums and slice states cleared
__global__ __launch_bounds__(kBfsBlock) void k_bfs_begin(BfsDev b, uint32_t sw)
{
    const uint32_t slice = blockIdx.x, cols = 64 * sw;
    for (uint32_t c = threadIdx.x; c < cols; c += blockDim.x) {
        const size_t i = (size_t)slice * cols + c;
        b.found[i] = 0;
        b.reach[i] = b.total[i] = 0;
        const bool in = (uint64_t)b.src0 + (uint64_t)slice * cols + c < b.src_end;
        const u64 m = __ballot(in);
        if (c % 64 == 0) b.live[(size_t)slice * sw + c / 64] = m;
    }
    if (threadIdx.x == 0) {
        b.done[slice] = b.levels[slice] = b.push[slice] = 0;
        b.front[slice] = 0;
    }
}

// Level 1: the frontier is the slice's sources, whose lists lie side by side.  One thread per
// arc (its source found by a binary search over the offsets in LDS), so hub sources spread
// over the grid.  Rows, visited and flags are zero before.
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_sources(BfsDev b, BfsLevel out)
{
    __shared__ uint32_t so[64 * SW + 1];
    const uint32_t slice = blockIdx.y, s0 = b.src0 + slice * 64 * SW;
    const uint32_t count = min(64u * SW, b.src_end - s0);
    for (uint32_t i = threadIdx.x; i <= count; i += blockDim.x) so[i] = b.off[s0 + i];
    __syncthreads();
    const uint64_t e1 = so[count];
    u64 *rows = out.rows + (size_t)slice * b.n * SW, *vis = b.visited + (size_t)slice * b.n * SW;
    for (uint64_t e = (uint64_t)so[0] + blockIdx.x * blockDim.x + threadIdx.x; e < e1; e += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = count;  // so[lo] <= e < so[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (so[mid] <= e) lo = mid; else hi = mid;
        }
        const uint32_t v = b.nbr[e];
        const size_t at = (size_t)v * SW + lo / 64;
        atomicOr(rows + at, 1ull << (lo % 64));
        atomicOr(vis + at, 1ull << (lo % 64));
        out.flag[(size_t)slice * b.npad + v] = 1;
    }
}

// The lanes of a team (SW / 2, two words of a row each) within its wavefront
template <int SW>
struct BfsTeam {
    static constexpr uint32_t L = SW / 2;
    uint32_t lane, tl, base;
    u64 mask;
    __device__ BfsTeam()
    {
        lane = threadIdx.x & 63u;
        tl = lane % L;
        base = lane - tl;
        mask = (L == 64 ? ~0ull : ((1ull << L) - 1)) << base;
    }
    __device__ bool any(bool p) const { return (__ballot(p) & mask) != 0; }
    __device__ bool all(bool p) const { return (__ballot(p) & mask) == mask; }
};

// got |= the frontier rows of in[0 .. len), this lane's two words; leaves once the team has
// every wanted bit.  The team reads L ids and their flags at a time and then the flagged
// rows, four loads in flight.
template <int SW>
__device__ __forceinline__ void bfs_pull_range(const BfsTeam<SW> &t, const uint32_t *__restrict__ in,
                                               uint32_t len, const uint8_t *__restrict__ flag,
                                               const ulonglong2 *__restrict__ rows, ulonglong2 want, ulonglong2 &got)
{
    constexpr uint32_t L = BfsTeam<SW>::L;
    // ids per trip: a narrow team takes several each, so that its loads overlap
    constexpr uint32_t K = L >= 4 ? 1 : 4 / L;
    for (uint32_t e = 0; e < len; e += L * K) {
        uint32_t id[K];
        bool f[K];
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) id[k] = e + k * L + t.tl < len ? in[e + k * L + t.tl] : ~0u;
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) f[k] = id[k] != ~0u && flag[id[k]];
        if constexpr (L == 1) {
#pragma unroll
            for (uint32_t k = 0; k < K; ++k)
                if (f[k]) {
                    const ulonglong2 r = rows[id[k]];
                    got.x |= r.x;
                    got.y |= r.y;
                }
        } else {
#pragma unroll
            for (uint32_t k = 0; k < K; ++k) {
                u64 m = __ballot(f[k]) & t.mask;
                while (m) {
                    uint32_t v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {  // past the last flagged id: the last again
                        v[q] = (uint32_t)__shfl((int)id[k], __ffsll(m) - 1);
                        if (m & (m - 1)) m &= m - 1;
                        else if (q == 3) m = 0;
                    }
                    ulonglong2 r[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) r[q] = rows[(size_t)v[q] * L + t.tl];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        got.x |= r[q].x;
                        got.y |= r[q].y;
                    }
                }
            }
        }
        if (t.all((want.x & ~got.x) == 0 && (want.y & ~got.y) == 0)) return;
    }
}

// the planes of two words (at index `at` in ulonglong2) whose sources `got` were found in
// `level`; `first`: none was found there before, so the planes hold nothing yet
__device__ __forceinline__ void bfs_keep(const BfsDev &b, size_t at, bool first, ulonglong2 got, uint32_t level)
{
#pragma unroll
    for (uint32_t k = 0; k < kBfsPlanes; ++k) {
        ulonglong2 *p = (ulonglong2 *)(b.plane + k * b.plane_stride) + at;
        const bool bit = (level >> k) & 1u;
        if (first) {
            *p = bit ? got : make_ulonglong2(0, 0);
        } else if (bit) {
            const ulonglong2 x = *p;
            *p = make_ulonglong2(x.x | got.x, x.y | got.y);
        }
    }
}

// a node's newly found sources: visited, its row (both at index `at` in ulonglong2), its flag
template <int SW>
__device__ __forceinline__ void bfs_found(const BfsDev &b, const BfsTeam<SW> &t, size_t at, u64 *rows, uint8_t *flag,
                                          ulonglong2 seen, ulonglong2 got, uint32_t level)
{
    const bool any = t.any((got.x | got.y) != 0);
    if (any) {
        ((ulonglong2 *)rows)[at] = got;
        ((ulonglong2 *)b.visited)[at] = make_ulonglong2(seen.x | got.x, seen.y | got.y);
        if (b.plane) bfs_keep(b, at, (seen.x | seen.y) == 0, got, level);
    }
    if (t.tl == 0) *flag = any ? 1 : 0;
}

// the planes after level 1, whose rows k_bfs_sources wrote
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_keep_first(BfsDev b, BfsLevel l)
{
    constexpr uint32_t L = SW / 2;
    const uint32_t slice = blockIdx.y;
    const uint64_t threads = (uint64_t)gridDim.x * kBfsBlock, all = (uint64_t)b.n * L;
    for (uint64_t i = (uint64_t)blockIdx.x * kBfsBlock + threadIdx.x; i < all; i += threads) {
        if (!l.flag[(size_t)slice * b.npad + i / L]) continue;
        const size_t at = (size_t)slice * b.n * L + i;
        bfs_keep(b, at, true, ((const ulonglong2 *)l.rows)[at], 1);
    }
}

// Push form of a level of rows of two words: the row of every node of the frontier, without the
// sources that have reached the head, ORed into the head's row, whose flag is set; k_bfs_pull
// then makes the flagged ones newly found nodes.  Rows and flags are zero before
// (k_bfs_count).  A wavefront takes 64 nodes, the arcs of the flagged ones side by side, a lane
// each; the lists of hubs come as tasks.
__global__ __launch_bounds__(kBfsBlock) void k_bfs_push(BfsDev b, BfsLevel prev, BfsLevel next, BfsDir dir)
{
    const uint32_t slice = blockIdx.y;
    if (b.done[slice] || !bfs_pushes<2>(b, slice, dir)) return;
    const size_t at = (size_t)slice * b.n, fat = (size_t)slice * b.npad;
    const uint8_t *flag = prev.flag + fat;
    const ulonglong2 *rows = (const ulonglong2 *)prev.rows + at;
    const uint32_t lane = threadIdx.x & 63u, waves = gridDim.x * (kBfsBlock / 64);
    const uint32_t wave = blockIdx.x * (kBfsBlock / 64) + threadIdx.x / 64;
    auto arc = [&](ulonglong2 r, uint32_t v) {
        const ulonglong2 seen = ((const ulonglong2 *)b.visited)[at + v];
        const u64 x = r.x & ~seen.x, y = r.y & ~seen.y;
        if (x) atomicOr(next.rows + 2 * (at + v), x);
        if (y) atomicOr(next.rows + 2 * (at + v) + 1, y);
        if (x | y) next.flag[fat + v] = 1;
    };
    for (uint64_t base = (uint64_t)wave * 64; base < b.n; base += (uint64_t)waves * 64) {
        const uint64_t u = base + lane;
        uint32_t e0 = 0, len = 0;
        if (u < b.n && flag[u]) {
            e0 = b.off[u];
            len = b.off[u + 1] - e0;
            if (len > kBfsHubDeg) len = 0;
        }
        if (!__ballot(len != 0)) continue;
        uint32_t end = len;  // of the lane's arcs among the wavefront's
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t below = __shfl_up(end, o);
            if (lane >= (uint32_t)o) end += below;
        }
        const uint32_t all = __shfl(end, 63);
        for (uint32_t i0 = 0; i0 < all; i0 += 64) {  // arc i0 + lane: of the first lane that ends past it
            const uint32_t i = i0 + lane;
            uint32_t j = 0;
#pragma unroll
            for (uint32_t step = 32; step; step >>= 1)
                if ((uint32_t)__shfl((int)end, (int)(j + step - 1)) <= i) j += step;
            j = min(j, 63u);
            const uint32_t first = __shfl(e0, (int)j) - (__shfl(end, (int)j) - __shfl(len, (int)j));
            if (i < all) arc(rows[base + j], b.nbr[(uint32_t)(first + i)]);
        }
    }
    for (uint32_t k = wave; k < b.tasks; k += waves) {
        const uint32_t u = b.task_node[k];
        if (!flag[u]) continue;
        const ulonglong2 r = rows[u];
        const uint32_t e0 = b.task_beg[k], len = b.task_end[k] - e0;
        for (uint32_t i = lane; i < len; i += 64) arc(r, b.nbr[(size_t)e0 + i]);
    }
}

// One level for the nodes with at most kBfsHubDeg tails: a team of SW / 2 lanes per node.
// After a push, what it left at every node.
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_pull(BfsDev b, BfsLevel prev, BfsLevel next, uint32_t level,
                                                        BfsDir dir)
{
    constexpr uint32_t L = SW / 2;
    const uint32_t slice = blockIdx.y;
    if (b.done[slice]) return;
    const BfsTeam<SW> t;
    const size_t at = (size_t)slice * b.n, fat = (size_t)slice * b.npad;
    const uint8_t *flag = prev.flag + fat;
    const ulonglong2 *rows = (const ulonglong2 *)prev.rows + at * L;
    const ulonglong2 live = ((const ulonglong2 *)b.live)[(size_t)slice * L + t.tl];
    const uint32_t teams = gridDim.x * (kBfsBlock / L);
    if constexpr (SW == 2)
        if (bfs_pushes<SW>(b, slice, dir)) {
            for (uint32_t v = blockIdx.x * kBfsBlock + threadIdx.x; v < b.n; v += teams)
                if (next.flag[fat + v])
                    bfs_found<SW>(b, t, at + v, next.rows, next.flag + fat + v, ((const ulonglong2 *)b.visited)[at + v],
                                  ((const ulonglong2 *)next.rows)[at + v], level);
            return;
        }
    for (uint32_t v = blockIdx.x * (kBfsBlock / L) + threadIdx.x / L; v < b.n; v += teams) {
        const uint32_t e0 = b.ioff[v], e1 = b.ioff[v + 1];
        if (e1 - e0 > kBfsHubDeg) continue;  // k_bfs_hub_tasks and k_bfs_hubs
        const size_t here = (at + v) * L + t.tl;
        const ulonglong2 seen = ((const ulonglong2 *)b.visited)[here];
        const ulonglong2 want = make_ulonglong2(live.x & ~seen.x, live.y & ~seen.y);
        ulonglong2 got = make_ulonglong2(0, 0);
        if (t.any((want.x | want.y) != 0)) bfs_pull_range<SW>(t, b.inbr + e0, e1 - e0, flag, rows, want, got);
        got.x &= want.x;
        got.y &= want.y;
        bfs_found<SW>(b, t, here, next.rows, next.flag + fat + v, seen, got, level);
    }
}

// The lists of hubs, cut into tasks: one wavefront per task, its teams every 64 / L-th run
// of ids, their words ORed into the task's row of `part`.
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_hub_tasks(BfsDev b, BfsLevel prev, BfsDir dir)
{
    constexpr uint32_t L = SW / 2, TEAMS = 64 / L;
    const uint32_t slice = blockIdx.y;
    if (b.done[slice] || bfs_pushes<SW>(b, slice, dir)) return;
    const BfsTeam<SW> t;
    const size_t at = (size_t)slice * b.n, fat = (size_t)slice * b.npad;
    const ulonglong2 live = ((const ulonglong2 *)b.live)[(size_t)slice * L + t.tl];
    const uint32_t waves = gridDim.x * (kBfsBlock / 64), team = t.lane / L;
    for (uint32_t k = blockIdx.x * (kBfsBlock / 64) + threadIdx.x / 64; k < b.tasks; k += waves) {
        const ulonglong2 seen = ((const ulonglong2 *)b.visited)[(at + b.task_node[k]) * L + t.tl];
        const ulonglong2 want = make_ulonglong2(live.x & ~seen.x, live.y & ~seen.y);
        if (!t.any((want.x | want.y) != 0)) continue;  // k_bfs_hubs does not read its row either
        const uint32_t e0 = b.task_beg[k], len = b.task_end[k] - e0, per = (len + TEAMS - 1) / TEAMS;
        const uint32_t lo = min(len, team * per), hi = min(len, lo + per);
        ulonglong2 got = make_ulonglong2(0, 0);
        bfs_pull_range<SW>(t, b.inbr + e0 + lo, hi - lo, prev.flag + fat, (const ulonglong2 *)prev.rows + at * L, want, got);
#pragma unroll
        for (uint32_t s = L; s < 64; s <<= 1) {
            got.x |= __shfl_xor(got.x, s);
            got.y |= __shfl_xor(got.y, s);
        }
        if (team == 0) ((ulonglong2 *)b.part)[((size_t)slice * b.tasks + k) * L + t.tl] = got;
    }
}

template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_hubs(BfsDev b, BfsLevel next, uint32_t level, BfsDir dir)
{
    constexpr uint32_t L = SW / 2;
    const uint32_t slice = blockIdx.y;
    if (b.done[slice] || bfs_pushes<SW>(b, slice, dir)) return;
    const BfsTeam<SW> t;
    const size_t at = (size_t)slice * b.n, fat = (size_t)slice * b.npad;
    const ulonglong2 live = ((const ulonglong2 *)b.live)[(size_t)slice * L + t.tl];
    const uint32_t teams = gridDim.x * (kBfsBlock / L);
    for (uint32_t h = blockIdx.x * (kBfsBlock / L) + threadIdx.x / L; h < b.hubs; h += teams) {
        const uint32_t v = b.hub_node[h];
        const size_t here = (at + v) * L + t.tl;
        const ulonglong2 seen = ((const ulonglong2 *)b.visited)[here];
        const ulonglong2 want = make_ulonglong2(live.x & ~seen.x, live.y & ~seen.y);
        ulonglong2 got = make_ulonglong2(0, 0);
        if (t.any((want.x | want.y) != 0))
            for (uint32_t k = b.hub_first[h]; k < b.hub_first[h + 1]; ++k) {
                const ulonglong2 r = ((const ulonglong2 *)b.part)[((size_t)slice * b.tasks + k) * L + t.tl];
                got.x |= r.x;
                got.y |= r.y;
            }
        got.x &= want.x;
        got.y &= want.y;
        bfs_found<SW>(b, t, here, next.rows, next.flag + fat + v, seen, got, level);
    }
}

// full adder over 64 columns at once
__device__ __forceinline__ void bfs_csa(u64 &hi, u64 &lo, u64 a, u64 b2, u64 c)
{
    const u64 u = a ^ b2;
    hi = (a & b2) | (u & c);
    lo = u ^ c;
}

// The newly found nodes of every source, per chunk of kBfsChunk nodes.  A thread adds one
// word of a chunk's rows, eight rows at a time, into bit-sliced counters (plane k holds bit
// k of 64 counts), then transposes the planes into 64 bytes: 13 operations per 64 bits
// added, where a ballot per column takes 256 per wavefront.
// Where the next level may push, the frontier before, which no kernel reads any more, is
// cleared here, so that the level finds its rows and flags zero.
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_count(BfsDev b, BfsLevel l, BfsLevel prev, bool clear)
{
    const uint32_t slice = blockIdx.y, chunks = bfs_chunks(b.n);
    if (b.done[slice]) return;
    const uint32_t w = threadIdx.x % SW;
    const size_t at = (size_t)slice * b.n;
    const uint32_t per_grid = gridDim.x * (kBfsBlock / SW);
    if (SW == 2 && clear) {
        ulonglong2 *pf = (ulonglong2 *)(prev.flag + (size_t)slice * b.npad);
        for (uint32_t i = blockIdx.x * kBfsBlock + threadIdx.x; i < b.npad / 16; i += gridDim.x * kBfsBlock) {
            const ulonglong2 f = pf[i];
            if (!(f.x | f.y)) continue;
            pf[i] = make_ulonglong2(0, 0);
            for (uint32_t k = 0; k < 16; ++k)
                if (((k < 8 ? f.x : f.y) >> (8 * (k % 8))) & 1u)
                    ((ulonglong2 *)prev.rows)[at + 16 * (size_t)i + k] = make_ulonglong2(0, 0);
        }
    }
    for (uint32_t c = blockIdx.x * (kBfsBlock / SW) + threadIdx.x / SW; c < chunks; c += per_grid) {
        u64 p[8] = {};
        const uint32_t v0 = c * kBfsChunk, v1 = min(b.n, v0 + kBfsChunk);
        bool any = false;
        auto add = [&](uint32_t v) {
            // eight flags of 0 or 1 as the low byte's bits, those past the last node dropped
            const u64 f8 = *(const u64 *)(l.flag + (size_t)slice * b.npad + v) & 0x0101010101010101ull;
            const uint32_t f = (uint32_t)((f8 * 0x0102040810204080ull) >> 56) & (0xffu >> (8 - min(8u, v1 - v)));
            if (!f) return;
            any = true;
            u64 x[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) x[k] = (f >> k) & 1u ? l.rows[(at + v + k) * SW + w] : 0ull;
            u64 two_a, two_b, four_a, four_b, eight;
            bfs_csa(two_a, p[0], p[0], x[0], x[1]);
            bfs_csa(two_b, p[0], p[0], x[2], x[3]);
            bfs_csa(four_a, p[1], p[1], two_a, two_b);
            bfs_csa(two_a, p[0], p[0], x[4], x[5]);
            bfs_csa(two_b, p[0], p[0], x[6], x[7]);
            bfs_csa(four_b, p[1], p[1], two_a, two_b);
            bfs_csa(eight, p[2], p[2], four_a, four_b);
#pragma unroll
            for (int k = 3; k < 8; ++k) {
                const u64 carry = p[k] & eight;
                p[k] ^= eight;
                eight = carry;
            }
        };
        if constexpr (SW == 2) {  // few threads: one round of loads finds the eights to add
            const ulonglong2 *q = (const ulonglong2 *)(l.flag + (size_t)slice * b.npad + v0);
            uint32_t eights = 0;
#pragma unroll
            for (uint32_t i = 0; i < kBfsChunk / 16; ++i) {
                const ulonglong2 f = q[i];
                eights |= (f.x ? 1u << (2 * i) : 0u) | (f.y ? 2u << (2 * i) : 0u);
            }
            for (; eights; eights &= eights - 1) {
                const uint32_t v = v0 + 8 * (uint32_t)(__ffs((int)eights) - 1);
                if (v < v1) add(v);
            }
        } else {
            for (uint32_t v = v0; v < v1; v += 8) add(v);
        }
        const size_t ci = (size_t)slice * chunks + c;
        if (w == 0) l.any[ci] = any ? 1 : 0;
        if (!any) continue;
        u64 *out = (u64 *)(l.count + (ci * SW + w) * 64);
#pragma unroll
        for (int q = 0; q < 8; ++q) {  // columns 8 q .. 8 q + 7: byte k of x from plane k, transposed
            u64 x = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) x |= ((p[k] >> (8 * q)) & 0xffull) << (8 * k);
            u64 s = (x ^ (x >> 7)) & 0x00AA00AA00AA00AAull;
            x ^= s ^ (s << 7);
            s = (x ^ (x >> 14)) & 0x0000CCCC0000CCCCull;
            x ^= s ^ (s << 14);
            s = (x ^ (x >> 28)) & 0x00000000F0F0F0F0ull;
            x ^= s ^ (s << 28);
            out[q] = x;
        }
    }
}

// the chunk counts summed per source into b.found: four columns per thread, the chunks
// split over blockIdx.x
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_totals(BfsDev b, BfsLevel l, uint32_t splits)
{
    constexpr uint32_t QUADS = 16 * SW;  // four columns each
    const uint32_t slice = blockIdx.y, chunks = bfs_chunks(b.n);
    if (b.done[slice]) return;
    for (uint32_t i = blockIdx.x * kBfsBlock + threadIdx.x; i < splits * QUADS; i += gridDim.x * kBfsBlock) {
        const uint32_t quad = i % QUADS, part = i / QUADS;
        uint32_t s[4] = {};
        for (uint32_t c = part; c < chunks; c += splits) {
            const size_t ci = (size_t)slice * chunks + c;
            if (!l.any[ci]) continue;
            const uint32_t x = ((const uint32_t *)l.count)[ci * QUADS + quad];
#pragma unroll
            for (int k = 0; k < 4; ++k) s[k] += (x >> (8 * k)) & 0xffu;
        }
        uint32_t *f = b.found + ((size_t)slice * QUADS + quad) * 4;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (s[k]) atomicAdd(f + k, s[k]);
    }
}

// The same for rows of two words, whose 32 quads leave k_bfs_totals few threads (18 us a level of
// a graph of a million nodes): eight parts of the chunks to a block, summed there before the
// atomics.  Also the arcs out of the chunks that hold a newly found node, a bound of the next
// frontier's.
__global__ __launch_bounds__(kBfsBlock) void k_bfs_totals_narrow(BfsDev b, BfsLevel l)
{
    constexpr uint32_t QUADS = 32, PARTS = kBfsBlock / QUADS;
    const uint32_t slice = blockIdx.y, chunks = bfs_chunks(b.n);
    if (b.done[slice]) return;
    __shared__ uint32_t red[PARTS][4 * QUADS];
    __shared__ u64 red_arcs[PARTS];
    const uint32_t quad = threadIdx.x % QUADS, part = threadIdx.x / QUADS, parts = gridDim.x * PARTS;
    uint32_t s[4] = {};
    u64 arcs = 0;
    for (uint32_t c = blockIdx.x * PARTS + part; c < chunks; c += parts) {
        const size_t ci = (size_t)slice * chunks + c;
        if (!l.any[ci]) continue;
        const uint32_t x = ((const uint32_t *)l.count)[ci * QUADS + quad];
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] += (x >> (8 * k)) & 0xffu;
        if (quad == 0) arcs += b.off[min(b.n, (c + 1) * kBfsChunk)] - b.off[c * kBfsChunk];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) red[part][4 * quad + k] = s[k];
    if (quad == 0) red_arcs[part] = arcs;
    __syncthreads();
    if (threadIdx.x < 4 * QUADS) {
        uint32_t t = 0;
        for (uint32_t p = 0; p < PARTS; ++p) t += red[p][threadIdx.x];
        if (t) atomicAdd(b.found + (size_t)slice * 4 * QUADS + threadIdx.x, t);
    } else if (threadIdx.x == 4 * QUADS) {
        u64 t = 0;
        for (uint32_t p = 0; p < PARTS; ++p) t += red_arcs[p];
        if (t) atomicAdd(b.front + slice, t);
    }
}

// end of a level, one block per slice: the per-source sums, the sources still searching, the
// form of the next level
template <int SW>
__global__ __launch_bounds__(1024) void k_bfs_level(BfsDev b, uint32_t level)
{
    const uint32_t slice = blockIdx.x;
    if (b.done[slice]) return;
    __shared__ uint32_t any;
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < 64 * SW; c += blockDim.x) {
        const size_t i = (size_t)slice * 64 * SW + c;
        const uint32_t f = b.found[i];
        b.found[i] = 0;
        b.reach[i] += f;
        b.total[i] += (u64)level * f;
        const u64 m = __ballot(f != 0);
        if (c % 64 == 0) {
            b.live[(size_t)slice * SW + c / 64] = m;
            if (m) any = 1;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (any) b.levels[slice] = level;
        else b.done[slice] = 1;
        if (SW == 2) {
            b.push[slice] = b.front[slice] <= b.push_arcs;
            b.front[slice] = 0;
        }
    }
}

// level into the distances of the found sources among the 8 of piece q of node v's row
template <int SW>
__device__ __forceinline__ void bfs_distance(const BfsDev &b, const BfsLevel &l, uint32_t slice, size_t v, uint32_t q,
                                             uint32_t level, uint16_t *dist)
{
    const uint32_t w = q / 8;
    const uint32_t bits = (uint32_t)(l.rows[((size_t)slice * b.n + v) * SW + w] >> (8 * (q % 8))) & 0xffu;
    if (!bits) return;
    uint4 *row = (uint4 *)(dist + (((size_t)slice * SW + w) * b.n + v) * 64) + q % 8;
    const uint4 x = *row;
    uint32_t r[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const uint32_t sh = 16u * (uint32_t)(h & 1);
        if ((bits >> h) & 1u) r[h >> 1] = (r[h >> 1] & ~(0xffffu << sh)) | (level << sh);
    }
    *row = make_uint4(r[0], r[1], r[2], r[3]);
}

// distances of the nodes found in the level, u16 [word][n][64]: a thread per 8 sources
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_dist(BfsDev b, BfsLevel l, uint32_t level, uint16_t *dist)
{
    const uint32_t slice = blockIdx.y;
    if (b.done[slice]) return;
    const uint64_t threads = (uint64_t)gridDim.x * kBfsBlock, all = (uint64_t)b.n * SW * 8;
    for (uint64_t i = (uint64_t)blockIdx.x * kBfsBlock + threadIdx.x; i < all; i += threads) {
        const uint32_t v = (uint32_t)(i / (SW * 8));
        if (l.flag[(size_t)slice * b.npad + v]) bfs_distance<SW>(b, l, slice, v, (uint32_t)(i % (SW * 8)), level, dist);
    }
}

// The same for rows of two words of a large graph, few of whose nodes are found in a level: a
// wavefront looks at 16 nodes at a time (11 us a level of a million nodes, 25 with a thread per 8
// sources; on a few thousand nodes 7 and 2)
__global__ __launch_bounds__(kBfsBlock) void k_bfs_dist_narrow(BfsDev b, BfsLevel l, uint32_t level, uint16_t *dist)
{
    constexpr uint32_t N = 16;
    const uint32_t slice = blockIdx.y;
    if (b.done[slice]) return;
    const uint32_t lane = threadIdx.x & 63u, step = gridDim.x * (kBfsBlock / 64) * N;
    for (uint64_t v0 = (blockIdx.x * (kBfsBlock / 64) + threadIdx.x / 64) * N; v0 < b.n; v0 += step) {
        const u64 found = __ballot(lane < N && v0 + lane < b.n && l.flag[(size_t)slice * b.npad + v0 + lane]);
        if (!found) continue;
        for (uint32_t i = lane; i < N * 16; i += 64)
            if ((found >> (i / 16)) & 1u) bfs_distance<2>(b, l, slice, v0 + i / 16, i % 16, level, dist);
    }
}

// the value of x in lane j (wave-uniform)
__device__ __forceinline__ double bfs_lane(double x, int j)
{
    const u64 b = (u64)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)b, j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), j);
    return __longlong_as_double((long long)(((u64)hi << 32) | lo));
}

// inv_sum[source] = Σ_{v=0..n-1} inv[d(v)] as the sequential f64 sum in node order rounds
// it, inv[d] = 1/d, from the kept levels.  One wavefront per source.
//
// A chain of n dependent adds takes 28 ns each.  But while the running sum stays within one
// binade [2^E, 2^(E+1)) its ulp is fixed, u = 2^(E-52), the sum is a multiple A u of it, and
// adding x rounds to A + round(x / u): a whole number that does not depend on A unless x / u
// lies halfway between two.  So a run of nodes adds Σ_d count_d round(2^.. / d) in any
// order as long as the result stays below 2^53 and no distance in it is a halfway case.
// The wavefront adds 64 chunks of kBfsChunk nodes at a time from the counts and their prefix
// sums; only a chunk in which the sum leaves its binade (some log2 n of them) or that holds a
// halfway case (the first binades) is replayed node by node.
// R-MAT-20, 2,048 sources: 0.87 ms, against 29.7 ms as chains.
template <int SW>
__global__ __launch_bounds__(kBfsBlock) void k_bfs_harmonic(BfsDev b, const uint8_t *__restrict__ count,
                                                            size_t count_stride, const uint8_t *__restrict__ any,
                                                            size_t any_stride, const double *__restrict__ inv,
                                                            uint32_t slices, double *__restrict__ out)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBfsBlock / 64) + threadIdx.x / 64);
    const uint32_t slice = wave / (64 * SW), col = wave % (64 * SW);
    if (slice >= slices || (uint64_t)b.src0 + wave >= b.src_end) return;
    const uint32_t levels = b.levels[slice], chunks = bfs_chunks(b.n);
    const size_t at = (size_t)slice * b.n, cat = (size_t)slice * chunks;
    // lane d - 1 holds 1/d and, for the current binade, round(x / u) and whether it is a tie
    const double x = lane < levels ? inv[lane + 1] : 0.0;
    const u64 xb = (u64)__double_as_longlong(x);
    const int xe = (int)(xb >> 52);  // biased exponent; 1/d is normal
    const u64 xm = (xb & ((1ull << 52) - 1)) | (1ull << 52);
    double acc = 0.0;
    for (uint32_t base = 0; base < chunks; base += 64) {
        const uint32_t c = base + lane;
        uint32_t cnt[(kBfsKeep + 3) / 4] = {};  // this lane's chunk: nodes at distance 1 .. levels, a byte each
#pragma unroll
        for (uint32_t d = 0; d < kBfsKeep; ++d)
            if (d < levels && c < chunks && any[d * any_stride + cat + c])
                cnt[d / 4] |= (uint32_t)count[d * count_stride + (cat + c) * 64 * SW + col] << (8 * (d % 4));
        uint32_t pos = 0;  // chunks base .. base + pos - 1 are in the sum
        const uint32_t end = min(64u, chunks - base);
        while (pos < end) {
            const u64 ab = (u64)__double_as_longlong(acc);
            const int ae = (int)(ab >> 52);
            const u64 am = (ab & ((1ull << 52) - 1)) | (1ull << 52);
            u64 q = 0;
            bool tie = false;
            if (lane < levels) {
                const int sh = ae - xe;
                if (acc == 0.0 || sh < 0) tie = true;  // leaves the binade at once
                else if (sh == 0) q = xm;
                else if (sh <= 53) {
                    const u64 half = 1ull << (sh - 1);
                    tie = (xm & (2 * half - 1)) == half;
                    q = (xm + half) >> sh;
                }
            }
            const u64 ties = __ballot(tie);
            u64 s = 0;
            bool stop = false;
#pragma unroll
            for (uint32_t d = 0; d < kBfsKeep; ++d)
                if (d < levels) {
                    const uint32_t k = (cnt[d / 4] >> (8 * (d % 4))) & 0xffu;
                    s += k * __shfl(q, (int)d);
                    stop = stop || (k && ((ties >> d) & 1u));
                }
            s = lane < pos || lane >= end ? 0ull : s < (1ull << 54) ? s : 1ull << 54;
            u64 sum = s;  // inclusive prefix; 64 terms of at most 2^54
#pragma unroll
            for (uint32_t o = 1; o < 64; o <<= 1) {
                const u64 y = __shfl_up(sum, o);
                if (lane >= o) sum += y;
            }
            stop = lane >= pos && lane < end && (stop || am + sum >= (1ull << 53));
            const u64 m = __ballot(stop);
            const uint32_t first = m ? (uint32_t)(__ffsll(m) - 1) : end;
            if (first > pos && acc != 0.0) {  // the sum before chunk `first`, an exact multiple of u
                const u64 a = am + __shfl(sum, (int)first - 1);
                acc = __longlong_as_double((long long)(((u64)ae << 52) | (a & ((1ull << 52) - 1))));
            }
            pos = first;
            if (first == end) break;
            // node by node: lane i takes nodes i and 64 + i of the chunk
            const uint32_t v0 = (base + first) * kBfsChunk;
#pragma unroll
            for (uint32_t h = 0; h < kBfsChunk; h += 64) {
                const uint32_t v = v0 + h + lane;
                const size_t word = (at + v) * SW + col / 64;
                uint32_t dist = 0;
                if (v < b.n && ((b.visited[word] >> (col % 64)) & 1ull))
#pragma unroll
                    for (uint32_t k = 0; k < kBfsPlanes; ++k)
                        dist |= (uint32_t)((b.plane[k * b.plane_stride + word] >> (col % 64)) & 1ull) << k;
                const double term = __shfl(x, (int)(dist ? dist - 1 : 0));
                u64 r = __ballot(dist != 0);
                while (r) {
                    acc = __dadd_rn(acc, bfs_lane(term, __ffsll(r) - 1));
                    r &= r - 1;
                }
            }
            ++pos;
        }
    }
    if (lane == 0) out[wave] = acc;
}

// The harmonic sums of searches of more than kBfsKeep levels, add by add:
// inv_sum[64 b + k] = Σ_{v=0..n-1} inv[dist_b[v][k]] as a sequential f64 sum in node
// order, dist_b = dist + b n 64 the distances of pass b of a group; inv[0] = 0
// (unreached), inv[d] = 1/d for d < entries.  One block per pass: the adds of a source
// are one dependent chain (lane k of wavefront 0 = source k), so the passes of a group
// run side by side, and the whole block streams the distances through LDS in tiles of
// kInvTile nodes -- tile t + 1 is loaded while tile t is summed -- so the summing
// wavefront never waits on HBM.  A 1/d table of at most kInvLds entries sits in LDS.
constexpr uint32_t kInvLds = 4096;
constexpr uint32_t kInvBlock = 256;
constexpr uint32_t kInvTile = 256;                    // nodes per tile: 32 KiB of u16 distances
constexpr uint32_t kInvVec = kInvTile * 64 * 2 / 16;  // uint4 per tile
constexpr uint32_t kInvPer = kInvVec / kInvBlock;     // uint4 per thread per tile

template <bool kLds>
__global__ __launch_bounds__(kInvBlock) void k_bfs_inv_sum(const uint16_t *__restrict__ dist,
                                                           const double *__restrict__ inv, uint32_t entries, uint32_t n,
                                                           const uint32_t *__restrict__ counts, double *out)
{
    __shared__ double tab[kLds ? kInvLds : 1];
    __shared__ uint4 tile[2][kInvVec];
    const uint32_t b = blockIdx.x, tid = threadIdx.x;
    if (kLds)
        for (uint32_t i = tid; i < entries; i += kInvBlock) tab[i] = inv[i];
    const uint4 *__restrict__ src = (const uint4 *)(dist + (size_t)b * n * 64);  // 8 uint4 per node
    const uint32_t tiles = (n + kInvTile - 1) / kInvTile;
    auto vecs = [&](uint32_t t) -> uint32_t {
        return (uint32_t)(std::min<uint64_t>(n, (uint64_t)(t + 1) * kInvTile) - (uint64_t)t * kInvTile) * 8u;
    };
    uint4 r[kInvPer];
    auto load = [&](uint32_t t) {
        const uint32_t m = vecs(t);
        const uint4 *p = src + (size_t)t * kInvVec;
#pragma unroll
        for (uint32_t j = 0; j < kInvPer; ++j) {
            const uint32_t i = tid + j * kInvBlock;
            if (i < m) r[j] = p[i];
        }
    };
    auto store = [&](uint32_t buf, uint32_t t) {
        const uint32_t m = vecs(t);
#pragma unroll
        for (uint32_t j = 0; j < kInvPer; ++j) {
            const uint32_t i = tid + j * kInvBlock;
            if (i < m) tile[buf][i] = r[j];
        }
    };
    double acc = 0.0;
    if (tiles) {
        load(0);
        store(0, 0);
    }
    __syncthreads();
    for (uint32_t t = 0; t < tiles; ++t) {
        if (t + 1 < tiles) load(t + 1);  // in flight while wavefront 0 sums tile t
        if (tid < 64) {
            const uint16_t *d = (const uint16_t *)tile[t & 1];
            const uint32_t m = vecs(t) / 8u;
            uint32_t j = 0;
            for (; j + 16 <= m; j += 16) {
                double x[16];
#pragma unroll
                for (uint32_t q = 0; q < 16; ++q) {
                    const uint16_t dv = d[(j + q) * 64 + tid];
                    x[q] = kLds ? tab[dv] : inv[dv];
                }
#pragma unroll
                for (uint32_t q = 0; q < 16; ++q) acc = __dadd_rn(acc, x[q]);
            }
            for (; j < m; ++j) {
                const uint16_t dv = d[j * 64 + tid];
                acc = __dadd_rn(acc, kLds ? tab[dv] : inv[dv]);
            }
        }
        if (t + 1 < tiles) store((t + 1) & 1, t + 1);
        __syncthreads();
    }
    if (tid < counts[b]) out[64 * b + tid] = acc;
}

// the tail of every arc, a wavefront per list
__global__ __launch_bounds__(kBfsBlock) void k_bfs_tails(const uint32_t *__restrict__ off, uint32_t n, uint32_t *tail)
{
    const uint32_t lane = threadIdx.x & 63u, waves = gridDim.x * (kBfsBlock / 64);
    for (uint32_t u = blockIdx.x * (kBfsBlock / 64) + threadIdx.x / 64; u < n; u += waves) {
        const uint32_t e1 = off[u + 1];
        for (uint64_t e = (uint64_t)off[u] + lane; e < e1; e += 64) tail[e] = u;
    }
}

// ioff from the ascending heads: for each of the n + 1 offsets the first arc whose head is not
// below it, by a binary search.  (Filled from the arcs instead, a long run of nodes without an
// arc to them is one thread's: a million of them took 32 ms.)
__global__ __launch_bounds__(kBfsBlock) void k_bfs_offsets(const uint32_t *__restrict__ head, uint32_t arcs, uint32_t n,
                                                           uint32_t *ioff)
{
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= n; v += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t lo = 0, len = arcs;
        while (len) {
            const uint32_t half = len / 2;
            if (head[(size_t)lo + half] < v) {
                lo += half + 1;
                len -= half + 1;
            } else {
                len = half;
            }
        }
        ioff[v] = lo;
    }
}

}  // namespace hb

namespace {
int efail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    hb::set_error(buf);
    return code;
}

struct Scoped {
    void *p = nullptr;
    ~Scoped() { release(); }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
};
}  // namespace

#define HBX_TRY(call)                                                                                    \
    do {                                                                                                 \
        const hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess)                                                                            \
            return efail(e_ == hipErrorOutOfMemory ? HB_ENOMEM : HB_EHIP, "hb_exact_bfs: %s failed: %s", \
                         #call, hipGetErrorString(e_));                                                  \
    } while (0)

namespace hb {
namespace {

constexpr uint64_t kBfsBudget = 16ull << 30;  // device memory of one group of slices
// What a group needs is kept between calls up to this much, one block per device: the driver
// clears freed device memory at some 40 GB/s before it hands it out again, so a call of 12 ms
// that takes and frees 5 GB soon waits 130 ms for it.  Given back when any allocation of the
// library fails (device_alloc) and by hb_release_memory.  A block in use belongs to one call; a
// second call at the same time takes memory of its own.
constexpr uint64_t kBfsHold = 2ull << 30;
constexpr int kBfsDevices = 16;

// SPARKX_HB_BFS_BYTES in the environment: a group of slices, and the reversed arcs, may take no
// more device memory than this (tests run several groups and the ways out of too little memory)
uint64_t bfs_limit()
{
    const char *e = getenv("SPARKX_HB_BFS_BYTES");
    return e ? strtoull(e, nullptr, 10) : UINT64_MAX;
}

struct BfsHeld {
    std::mutex mu;
    void *p[kBfsDevices] = {};
    size_t bytes[kBfsDevices] = {};
} g_bfs_held;

struct BfsMemory {
    void *p = nullptr;
    size_t bytes = 0;
    int device = -1;
    hipStream_t stream = nullptr;

    explicit BfsMemory(hipStream_t s) : stream(s) {}
    ~BfsMemory() { release(); }
    hipError_t take(size_t want)
    {
        if (want > bfs_limit()) return hipErrorOutOfMemory;
        if (device < 0) {
            const hipError_t e = hipGetDevice(&device);
            if (e != hipSuccess) return e;
        }
        if (device < kBfsDevices) {
            std::lock_guard<std::mutex> lock(g_bfs_held.mu);
            void *&held = g_bfs_held.p[device];
            if (held && g_bfs_held.bytes[device] >= want) {
                p = held;
                bytes = g_bfs_held.bytes[device];
                held = nullptr;
                return hipSuccess;
            }
            if (held) (void)hipFree(held);  // too small: its place is for this one
            held = nullptr;
        }
        const hipError_t e = device_alloc(&p, want);
        if (e != hipSuccess) p = nullptr;
        else bytes = want;
        return e;
    }
    void release()
    {
        if (!p) return;
        (void)hipStreamSynchronize(stream);  // also where a call ends with an error
        if (device < kBfsDevices && bytes <= kBfsHold) {
            std::lock_guard<std::mutex> lock(g_bfs_held.mu);
            if (!g_bfs_held.p[device]) {
                g_bfs_held.p[device] = p;
                g_bfs_held.bytes[device] = bytes;
                p = nullptr;
                return;
            }
        }
        (void)hipFree(p);
        p = nullptr;
    }
};

// How a group of searches runs: kSums counts only; kKeep keeps distances and counts for
// k_bfs_harmonic; kLong records u16 distances for k_bfs_inv_sum
enum class BfsMode { kSums, kKeep, kLong };

// the group's one allocation, cut up
struct BfsPlan {
    uint32_t sw = 0, slices = 0;
    uint32_t words = 0;  // of a row that hold sources: sw, or 1 of 2 where the distances of both do not fit
    size_t rows_stride = 0, flag_stride = 0, count_stride = 0, any_stride = 0;  // per level
    uint32_t counts = 0;  // count buffers; rows and flags have two, by level parity
    size_t bytes = 0;
    size_t o_vis = 0, o_rows = 0, o_flag = 0, o_count = 0, o_any = 0, o_part = 0, o_plane = 0, o_dist = 0, o_src = 0;
    bool keep = false;
};

BfsPlan bfs_plan(uint32_t n, uint32_t tasks, uint32_t sw, uint32_t words, uint32_t slices, BfsMode mode)
{
    BfsPlan p;
    p.sw = sw;
    p.words = words;
    p.slices = slices;
    p.keep = mode == BfsMode::kKeep;
    p.counts = p.keep ? kBfsKeep : 1;
    const size_t chunks = (n + kBfsChunk - 1) / kBfsChunk, npad = chunks * kBfsChunk;
    auto take = [&](size_t bytes) {
        const size_t at = p.bytes;
        p.bytes += (bytes + 255) & ~(size_t)255;
        return at;
    };
    p.rows_stride = (size_t)slices * n * sw;
    p.flag_stride = (size_t)slices * npad;
    p.any_stride = (size_t)slices * chunks;
    p.count_stride = p.any_stride * 64 * sw;
    p.o_vis = take(p.rows_stride * 8);
    p.o_rows = take(p.rows_stride * 8 * 2);
    p.o_flag = take(p.flag_stride * 2);
    p.o_plane = take(p.keep ? p.rows_stride * 8 * kBfsPlanes : 0);
    p.o_count = take(p.count_stride * p.counts);
    p.o_any = take(p.any_stride * p.counts);
    p.o_part = take((size_t)slices * tasks * sw * 8);
    p.o_dist = take(mode == BfsMode::kLong ? (size_t)slices * n * words * 128 : 0);
    // per source: reach, total, sum, found; per word: live, source count; per slice: front, done,
    // levels, push
    p.o_src = take((size_t)slices * (sw * (64 * 28 + 12) + 20));
    return p;
}

struct BfsGroup {
    BfsDev b{};
    BfsLevel level0{};
    BfsPlan plan;
    uint16_t *dist = nullptr;
    double *sums = nullptr;
    uint32_t *word_count = nullptr;

    BfsLevel level(uint32_t l) const  // of level l >= 1
    {
        const uint32_t i = (l - 1) % 2, c = (l - 1) % plan.counts;
        return {level0.rows + i * plan.rows_stride, level0.flag + i * plan.flag_stride,
                level0.count + c * plan.count_stride, level0.any + c * plan.any_stride};
    }
    void place(char *base, const BfsPlan &p)
    {
        plan = p;
        const size_t src = (size_t)p.slices * 64 * p.sw, words = (size_t)p.slices * p.sw;
        b.visited = (u64 *)(base + p.o_vis);
        level0 = {(u64 *)(base + p.o_rows), (uint8_t *)(base + p.o_flag), (uint8_t *)(base + p.o_count),
                  (uint8_t *)(base + p.o_any)};
        b.part = (u64 *)(base + p.o_part);
        b.plane = p.keep ? (u64 *)(base + p.o_plane) : nullptr;
        b.plane_stride = p.rows_stride;
        dist = (uint16_t *)(base + p.o_dist);
        b.reach = (u64 *)(base + p.o_src);
        b.total = b.reach + src;
        sums = (double *)(b.total + src);
        b.live = (u64 *)(sums + src);
        b.front = b.live + words;
        b.found = (uint32_t *)(b.front + p.slices);
        word_count = b.found + src;
        b.done = word_count + words;
        b.levels = b.done + p.slices;
        b.push = b.levels + p.slices;
    }
};

unsigned bfs_grid(uint64_t threads, uint32_t slices)
{
    const uint64_t cap = std::max<uint64_t>(512, 16384 / slices);
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((threads + kBfsBlock - 1) / kBfsBlock, cap));
}

// levels from .. to of every slice; returns at once where a slice is done
template <int SW>
hipError_t bfs_levels(const BfsGroup &g, uint32_t from, uint32_t to, uint64_t source_arcs, BfsMode mode, BfsDir dir,
                      hipStream_t s)
{
    const BfsDev &b = g.b;
    const uint32_t slices = g.plan.slices, chunks = (b.n + kBfsChunk - 1) / kBfsChunk;
    const uint32_t splits = std::min(chunks, std::max(1u, 256u / slices));
    for (uint32_t l = from; l <= to; ++l) {
        const BfsLevel next = g.level(l);
        if (l == 1) {
            k_bfs_sources<SW><<<dim3(bfs_grid(source_arcs, slices), slices), kBfsBlock, 0, s>>>(b, next);
            if (b.plane)
                k_bfs_keep_first<SW><<<dim3(bfs_grid((uint64_t)b.n * (SW / 2), slices), slices), kBfsBlock, 0, s>>>(b, next);
        } else {
            const BfsLevel prev = g.level(l - 1);
            if (SW == 2 && dir != BfsDir::kPull)
                k_bfs_push<<<dim3(std::min(bfs_grid(b.n, slices), 1024u), slices), kBfsBlock, 0, s>>>(b, prev, next, dir);
            k_bfs_pull<SW><<<dim3(bfs_grid((uint64_t)b.n * (SW / 2), slices), slices), kBfsBlock, 0, s>>>(b, prev, next, l,
                                                                                                      dir);
            if (b.tasks && dir != BfsDir::kPush) {
                k_bfs_hub_tasks<SW><<<dim3(bfs_grid((uint64_t)b.tasks * 64, slices), slices), kBfsBlock, 0, s>>>(b, prev,
                                                                                                              dir);
                k_bfs_hubs<SW><<<dim3(bfs_grid((uint64_t)b.hubs * (SW / 2), slices), slices), kBfsBlock, 0, s>>>(b, next, l,
                                                                                                             dir);
            }
        }
        k_bfs_count<SW><<<dim3(bfs_grid((uint64_t)chunks * SW, slices), slices), kBfsBlock, 0, s>>>(
            b, next, g.level(l > 1 ? l - 1 : 2), dir != BfsDir::kPull && l > 1);
        if (SW == 2)
            k_bfs_totals_narrow<<<dim3(std::min((chunks + 7) / 8, std::max(1u, 128u / slices)), slices), kBfsBlock, 0, s>>>(
                b, next);
        else
            k_bfs_totals<SW><<<dim3(bfs_grid((uint64_t)splits * 16 * SW, slices), slices), kBfsBlock, 0, s>>>(b, next,
                                                                                                          splits);
        k_bfs_level<SW><<<slices, std::min(1024, 64 * SW), 0, s>>>(b, l);
        // a level that found nothing has marked its slice done and records nothing
        if (mode == BfsMode::kLong) {
            if (SW == 2 && b.n >= 1u << 17)
                k_bfs_dist_narrow<<<dim3(bfs_grid((uint64_t)b.n * 4, slices), slices), kBfsBlock, 0, s>>>(b, next, l, g.dist);
            else
                k_bfs_dist<SW><<<dim3(bfs_grid((uint64_t)b.n * SW * 8, slices), slices), kBfsBlock, 0, s>>>(b, next, l, g.dist);
        }
    }
    return hipGetLastError();
}

// The reversed CSR of directed arcs, offsets then tails, into `rev`, its offsets also to the host.
// A stable sort by head (4M arcs: 0.3 ms; counting and placing them with atomics took 2); short of
// memory nothing is kept.
hipError_t bfs_reverse(const uint32_t *off, const uint32_t *nbr, uint32_t n, uint32_t arcs, Scoped &rev,
                       std::vector<uint32_t> &h_ioff, hipStream_t s)
{
#define HB_REV_TRY(call)                   \
    do {                                   \
        const hipError_t e_ = (call);      \
        if (e_ != hipSuccess) {            \
            (void)hipStreamSynchronize(s); \
            rev.release();                 \
            return e_;                     \
        }                                  \
    } while (0)
    Scoped tmp;
    const unsigned bits = std::max(1u, 32u - (unsigned)__builtin_clz(std::max(n - 1, 1u)));
    size_t bytes = 0;
    HB_REV_TRY(rocprim::radix_sort_pairs(nullptr, bytes, nbr, (uint32_t *)nullptr, (uint32_t *)nullptr,
                                         (uint32_t *)nullptr, (size_t)arcs, 0, bits, s));
    const size_t words = (bytes + 255) / 4 / 64 * 64;
    const size_t rev_bytes = ((size_t)n + 1 + arcs) * 4, tmp_bytes = (words + 2 * (size_t)arcs) * 4;
    if (rev_bytes + tmp_bytes > bfs_limit()) return hipErrorOutOfMemory;
    HB_REV_TRY(device_alloc(&rev.p, rev_bytes));
    HB_REV_TRY(device_alloc(&tmp.p, tmp_bytes));
    uint32_t *ioff = (uint32_t *)rev.p, *inbr = ioff + n + 1;
    uint32_t *tail = (uint32_t *)tmp.p + words, *head = tail + arcs;
    k_bfs_tails<<<(unsigned)std::min<uint64_t>(((uint64_t)n + 3) / 4, 16384), kBfsBlock, 0, s>>>(off, n, tail);
    HB_REV_TRY(rocprim::radix_sort_pairs(tmp.p, bytes, nbr, head, tail, inbr, (size_t)arcs, 0, bits, s));
    k_bfs_offsets<<<(unsigned)std::min<uint64_t>((uint64_t)n / kBfsBlock + 1, 16384), kBfsBlock, 0, s>>>(head, arcs, n, ioff);
    HB_REV_TRY(hipGetLastError());
    h_ioff.resize((size_t)n + 1);
    HB_REV_TRY(hipMemcpyAsync(h_ioff.data(), ioff, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost, s));
    HB_REV_TRY(hipStreamSynchronize(s));
#undef HB_REV_TRY
    return hipSuccess;
}

// nodes with long lists and the tasks those are cut into (hub h: tasks first[h] ..)
struct BfsHubs {
    std::vector<uint32_t> node, first, tnode, tbeg, tend;

    BfsHubs(const uint32_t *off, uint32_t n)
    {
        for (uint64_t v0 = 0; v0 < n; v0 += 16) {  // most runs of 16 hold none (one vector loop)
            const uint32_t v1 = (uint32_t)std::min<uint64_t>(n, v0 + 16);
            uint32_t any = 0;
            for (uint32_t v = (uint32_t)v0; v < v1; ++v) any |= off[v + 1] - off[v] > kBfsHubDeg;
            if (!any) continue;
            for (uint32_t v = (uint32_t)v0; v < v1; ++v)
                if (off[v + 1] - off[v] > kBfsHubDeg) cut(v, off[v], off[v + 1]);
        }
        first.push_back((uint32_t)tnode.size());
    }

private:
    void cut(uint32_t v, uint64_t beg, uint64_t end)
    {
        node.push_back(v);
        first.push_back((uint32_t)tnode.size());
        for (uint64_t e = beg; e < end; e += kBfsHubArcs) {
            tnode.push_back(v);
            tbeg.push_back((uint32_t)e);
            tend.push_back((uint32_t)std::min<uint64_t>(e + kBfsHubArcs, end));
        }
    }
};

}  // namespace

void release_held()
{
    std::lock_guard<std::mutex> lock(g_bfs_held.mu);
    for (void *&p : g_bfs_held.p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
}

hipError_t device_alloc(void **p, size_t bytes)
{
    *p = nullptr;
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        release_held();
        e = hipMalloc(p, bytes);
        if (e != hipSuccess) (void)hipGetLastError();
    }
    if (e != hipSuccess) *p = nullptr;
    return e;
}

int exact_bfs(const uint32_t *off, const uint32_t *h_off, const uint32_t *nbr, uint32_t n, bool symmetric,
              uint64_t s_begin,
              uint64_t s_end, uint64_t *reach, uint64_t *total, double *inv_sum, hipStream_t s)
{
    if (s_begin > s_end || s_end > n) return efail(HB_EINVAL, "hb_exact_bfs: sources [%llu, %llu) outside [0, %u)",
                                                   (unsigned long long)s_begin, (unsigned long long)s_end, n);
    if (s_begin == s_end) return HB_OK;
    const uint32_t arcs = h_off[n];
    BfsGroup g;
    BfsDev &b = g.b;
    b.off = off;
    b.nbr = nbr;
    b.n = n;
    b.npad = (n + kBfsChunk - 1) / kBfsChunk * kBfsChunk;
    // tails of the arcs to each node: the lists themselves, or the reversed arcs; directed graphs
    // with few sources, and those whose reversed arcs find no memory, only push
    Scoped rev;
    std::vector<uint32_t> h_ioff;
    b.ioff = off;
    b.inbr = nbr;
    const bool directed = !symmetric && arcs != 0;
    bool push_only = directed && s_end - s_begin <= kBfsFew;
    if (directed && !push_only) {
        const hipError_t e = bfs_reverse(off, nbr, n, arcs, rev, h_ioff, s);
        if (e == hipSuccess) {
            b.ioff = (const uint32_t *)rev.p;
            b.inbr = b.ioff + n + 1;
        } else if (e == hipErrorOutOfMemory) {
            push_only = true;
        } else {
            HBX_TRY(e);
        }
    }
    // hubs and their tasks, of the lists that pulls read or, where there are none, those that pushes do
    Scoped hub;
    {
        const BfsHubs h(h_ioff.empty() ? h_off : h_ioff.data(), n);
        b.hubs = (uint32_t)h.node.size();
        b.tasks = (uint32_t)h.tnode.size();
        if (b.hubs) {
            std::vector<uint32_t> all;
            for (const auto *v : {&h.node, &h.first, &h.tnode, &h.tbeg, &h.tend}) all.insert(all.end(), v->begin(), v->end());
            HBX_TRY(device_alloc(&hub.p, all.size() * 4));
            HBX_TRY(hipMemcpy(hub.p, all.data(), all.size() * 4, hipMemcpyHostToDevice));
            b.hub_node = (const uint32_t *)hub.p;
            b.hub_first = b.hub_node + b.hubs;
            b.task_node = b.hub_first + b.hubs + 1;
            b.task_beg = b.task_node + b.tasks;
            b.task_end = b.task_beg + b.tasks;
        }
    }
    // both read the same lists, which the tasks are of
    const bool may_push = push_only || (symmetric && arcs >= kBfsPushArcs);
    b.push_arcs = arcs / kBfsPush;
    BfsMode mode = inv_sum ? BfsMode::kKeep : BfsMode::kSums;
    Scoped inv;
    BfsMemory mem(s);
    std::vector<double> h_inv(1, 0.0);  // 1/d as correctly rounded host divisions; entry 0: unreached
    auto inverses = [&](uint32_t levels) -> int {
        if (inv.p && h_inv.size() > levels) return HB_OK;
        for (size_t d = h_inv.size(); d <= levels; ++d) h_inv.push_back(1.0 / (double)d);
        inv.release();
        HBX_TRY(device_alloc(&inv.p, h_inv.size() * 8));
        HBX_TRY(hipMemcpyAsync(inv.p, h_inv.data(), h_inv.size() * 8, hipMemcpyHostToDevice, s));
        return HB_OK;
    };
    for (uint64_t s0 = s_begin; s0 < s_end;) {
        if (!mem.p) {
            // the widest rows and then the most slices that fit into memory that is kept, with
            // rows of at least 64 bytes (half a cache line), else into the budget
            const uint64_t words = (s_end - s0 + 63) / 64;
            auto bytes = [&](uint32_t w, uint32_t k) { return (uint64_t)bfs_plan(n, b.tasks, w, w, k, mode).bytes; };
            uint32_t wide = 2;
            while (wide < 32 && wide < words && !push_only) wide *= 2;
            uint32_t sw = wide;
            uint64_t budget = std::min(kBfsHold, bfs_limit());
            while (sw > 8 && bytes(sw, 1) > budget) sw /= 2;
            if (bytes(sw, 1) > budget) {
                sw = wide;
                budget = std::min(kBfsBudget, bfs_limit());
                while (sw > 2 && bytes(sw, 1) > budget) sw /= 2;
            }
            uint32_t slices = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((words + sw - 1) / sw, budget / bytes(sw, 1)));
            while (slices > 1 && bytes(sw, slices) > budget) --slices;
            for (uint32_t row = sw;;) {
                const BfsPlan p = bfs_plan(n, b.tasks, sw, row, slices, mode);
                const hipError_t e = mem.take(p.bytes);
                if (e == hipSuccess) {
                    g.place((char *)mem.p, p);
                    break;
                }
                if (e != hipErrorOutOfMemory) HBX_TRY(e);
                if (slices > 1) slices /= 2;
                else if (sw > 2) row = sw /= 2;
                else if (mode == BfsMode::kLong && row == 2) row = 1;
                else HBX_TRY(e);
            }
        }
        const uint32_t per_slice = 64 * g.plan.words;
        // the last group may need fewer slices; the buffers keep their strides
        const uint32_t slices = (uint32_t)std::min<uint64_t>(g.plan.slices, (s_end - s0 + per_slice - 1) / per_slice);
        BfsGroup r = g;
        r.plan.slices = slices;
        r.b.src0 = (uint32_t)s0;
        const uint64_t group_end = std::min<uint64_t>(s_end, s0 + (uint64_t)slices * per_slice);
        r.b.src_end = (uint32_t)group_end;
        uint64_t source_arcs = 0;
        for (uint32_t i = 0; i < slices; ++i) {
            const uint64_t a = s0 + (uint64_t)i * per_slice, e = std::min<uint64_t>(a + per_slice, s_end);
            source_arcs = std::max<uint64_t>(source_arcs, h_off[e] - h_off[a]);
        }
        const uint64_t row_words = (uint64_t)slices * n * g.plan.sw;
        const unsigned zgrid = (unsigned)std::min<uint64_t>((row_words / 2 + kBfsBlock - 1) / kBfsBlock, 16384);
        k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.b.visited, row_words / 2);
        k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.level(1).rows, row_words / 2);
        k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.level(1).flag, (uint64_t)slices * r.b.npad / 16);
        if (may_push && r.plan.sw == 2) {  // level 2 too finds them zero
            k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.level(2).rows, row_words / 2);
            k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.level(2).flag, (uint64_t)slices * r.b.npad / 16);
        }
        if (mode == BfsMode::kLong) k_bfs_zero<uint4><<<zgrid, kBfsBlock, 0, s>>>((uint4 *)r.dist, (uint64_t)slices * n * g.plan.words * 8);
        k_bfs_begin<<<slices, kBfsBlock, 0, s>>>(r.b, r.plan.sw);
        // launches past a slice's last level return at once, so the host looks every 4, 8, ..
        // levels only
        std::vector<uint32_t> state(3 * (size_t)g.plan.slices);
        uint32_t at = 0;  // levels launched
        bool all = false, each = false;
        while (!all) {
            uint32_t to = at + (at < 8 ? 4 : std::min(64u, at / 2));
            if (mode == BfsMode::kKeep) to = std::min(to, kBfsKeep);
            if (mode == BfsMode::kLong) to = std::min(to, 65535u);
            if (to == at) break;
            // Past the eighth level, where a frontier seldom grows at a stroke, the levels up to the
            // next look push without being asked if all slices were to push at this one
            BfsDir dir = BfsDir::kPull;
            if (may_push && r.plan.sw == 2) dir = push_only || (at >= 8 && each) ? BfsDir::kPush : BfsDir::kEither;
            if (dir == BfsDir::kPush) to = std::min(to, at + 16);
            hipError_t e = hipErrorInvalidValue;
            switch (r.plan.sw) {
            case 2: e = bfs_levels<2>(r, at + 1, to, source_arcs, mode, dir, s); break;
            case 4: e = bfs_levels<4>(r, at + 1, to, source_arcs, mode, dir, s); break;
            case 8: e = bfs_levels<8>(r, at + 1, to, source_arcs, mode, dir, s); break;
            case 16: e = bfs_levels<16>(r, at + 1, to, source_arcs, mode, dir, s); break;
            case 32: e = bfs_levels<32>(r, at + 1, to, source_arcs, mode, dir, s); break;
            }
            HBX_TRY(e);
            HBX_TRY(hipMemcpyAsync(state.data(), r.b.done, state.size() * 4, hipMemcpyDeviceToHost, s));
            HBX_TRY(hipStreamSynchronize(s));
            at = to;
            all = true;
            each = true;
            for (uint32_t i = 0; i < slices; ++i) {
                all = all && state[i];
                each = each && (state[i] || state[2 * (size_t)g.plan.slices + i]);
            }
        }
        if (!all && mode == BfsMode::kKeep) {  // long searches: this group again, and the rest, by distances
            mode = BfsMode::kLong;
            mem.release();
            continue;
        }
        if (!all)
            return efail(HB_ERANGE, "hb_exact_bfs: eccentricity above 65535 (harmonic sums need u16 distances)");
        const size_t sources = (size_t)(group_end - s0);
        const size_t cols = (size_t)g.plan.slices * 64 * g.plan.sw;
        std::vector<u64> h_sums(2 * cols);
        if (reach || total)
            HBX_TRY(hipMemcpyAsync(h_sums.data(), r.b.reach, h_sums.size() * 8, hipMemcpyDeviceToHost, s));
        if (inv_sum) {
            uint32_t levels = 0;
            for (uint32_t i = 0; i < slices; ++i) levels = std::max(levels, state[g.plan.slices + i]);
            if (int rc = inverses(std::max(levels, kBfsKeep))) return rc;
            if (mode == BfsMode::kKeep) {
                const BfsPlan &p = g.plan;
                const unsigned grid = (unsigned)((sources + kBfsBlock / 64 - 1) / (kBfsBlock / 64));
#define HB_BFS_HARMONIC(SW)                                                                                       \
    case SW:                                                                                                      \
        k_bfs_harmonic<SW><<<grid, kBfsBlock, 0, s>>>(r.b, r.level0.count, p.count_stride, r.level0.any, p.any_stride, \
                                                      (const double *)inv.p, slices, r.sums);                      \
        break;
                switch (p.sw) { HB_BFS_HARMONIC(2) HB_BFS_HARMONIC(4) HB_BFS_HARMONIC(8) HB_BFS_HARMONIC(16) HB_BFS_HARMONIC(32) }
#undef HB_BFS_HARMONIC
            } else {
                const uint32_t passes = (uint32_t)((sources + 63) / 64);
                std::vector<uint32_t> counts(passes, 64u);
                counts.back() = (uint32_t)(sources - (size_t)(passes - 1) * 64);
                HBX_TRY(hipMemcpyAsync(r.word_count, counts.data(), passes * 4, hipMemcpyHostToDevice, s));
                HBX_TRY(hipStreamSynchronize(s));  // `counts` is a pageable host buffer
                const uint32_t entries = levels + 1;
                if (entries <= kInvLds)
                    k_bfs_inv_sum<true><<<passes, kInvBlock, 0, s>>>(r.dist, (const double *)inv.p, entries, n,
                                                                     r.word_count, r.sums);
                else
                    k_bfs_inv_sum<false><<<passes, kInvBlock, 0, s>>>(r.dist, (const double *)inv.p, entries, n,
                                                                      r.word_count, r.sums);
            }
            HBX_TRY(hipGetLastError());
            HBX_TRY(hipMemcpyAsync(inv_sum + (s0 - s_begin), r.sums, sources * 8, hipMemcpyDeviceToHost, s));
        }
        HBX_TRY(hipStreamSynchronize(s));
        for (size_t i = 0; i < sources; ++i) {
            if (reach) reach[s0 - s_begin + i] = h_sums[i];
            if (total) total[s0 - s_begin + i] = h_sums[cols + i];
        }
        s0 = group_end;
    }
    return HB_OK;
}

}  // namespace hb
