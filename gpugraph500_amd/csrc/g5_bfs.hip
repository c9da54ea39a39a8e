// g5_bfs.hip -- single-root local expansion: the GPU "Derived" plug-in of
// GlobalBFS (cpu_2d/cuda/cuda_bfs.h:39-84) re-designed for gfx950.
//
// State per search lives in HBM as bitmaps (visited, out) plus a sorted
// uint32 in-queue.  A level is:
//   1. the frontier's bitmap -> sorted queue with its degree prefix (two
//      launches; a queue that the host gives gets its prefix by a scan),
//   2. k_expand: edge-balanced top-down expansion -- every block takes a
//      1024-edge tile of the level's edge range, finds each edge's source by
//      binary search among the tile's, staged in LDS, and for an unvisited target sets
//      its out bit (atomicOr, skipped when already set) and lowers its parent
//      with atomicMin.  The surviving parent is the minimum-id frontier
//      neighbour: the same vertex CPUBFS_bin's ascending scan keeps
//      (cpu_2d/cpubfs_bin.cpp:150-173), independent of thread timing.
//   3. k_commit: visited |= out, level := depth + 1, sums of the new vertices
//      and their degrees per bitmap tile, which step 1 starts from.
// Every counter that the host reads is a sum per workgroup, added up by one
// more workgroup that writes it to pinned memory (same-address atomics take
// their turns, and a copy costs a launch and more).  Queues are born sorted and unique, so the reference's thrust::sort and host
// unique_copy (cuda_bfs.cu:380-475) have no counterpart.
//
// g5_bfs_run (1x1 block, resident) also runs dense levels bottom-up: each
// unvisited vertex scans its sorted neighbour list and stops at the first
// frontier vertex, which is again the minimum-id frontier neighbour, so both
// directions give identical parents and levels.  Its levels are one kernel
// each and decided on the device (k_level); with the codec, with accounting or
// with a forced direction the host drives them from the level's counters
// (k_expand and k_commit, or k_bottom_up, which commits as it goes, and the
// sorted queue of step 1 where a top-down level or the codec needs it).  The
// hooks leave the row frontier a bitmap until a top-down level needs it.  The
// codec's whole search at scale 22 takes 664 us (1391 with 128 launches; now
// 55), a 2 x 2 grid's on one card 3.3 ms (6.5; 641 launches, now 271).
#include <algorithm>

#include "g5_codec.hpp"
#include "g5_internal.hpp"

namespace {

constexpr uint32_t kNoParent = 0xFFFFFFFFu;
constexpr uint32_t kRootMark = 0xFFFFFFFEu;  // parent slot of the root column
constexpr int kExpandBlock = 256;
constexpr int kExpandTile = 1024;            // edges per block tile
constexpr int kExpandGrid = 4096;            // persistent grid, grid-stride over tiles
constexpr int kTileSrc = 512;                // sources of a tile that are staged in LDS
constexpr int kParts = 4096;                 // workgroups that leave a sum each, at most

// kNewEdges: degree sum of the newly reached vertices (1x1 only); kBuEdges,
// kBuVerts: neighbours checked and vertices scanned by a bottom-up level;
// kCodecErr: set when a level queue's codec round trip failed (g5_bfs_run)
enum Cnt {
    kQLen = 0, kEdges = 1, kNew = 2, kOutLen = 3, kNewEdges = 4, kBuEdges = 5, kBuVerts = 6, kCodecErr = 7, kNCnt = 8
};
// direction switch of the 1x1 search (Beamer, Asanovic, Patterson, SC'12):
// top-down -> bottom-up when the frontier's edges exceed the unexplored
// edges / alpha, back when the frontier holds fewer than n / beta vertices
// (g5_bfs_tune).  As in the GAP benchmark's implementation of the rule, the
// unexplored edges are reduced only by the frontiers expanded top-down, so
// that the few vertices left at the tail of the search do not flip it back
// to bottom-up, where every unreached vertex would be scanned again.
// alpha 20: 3.32 ms per root at scale 26 against 3.51 ms with 14 and 3.94
// with 8 (scale 22: within 1 %); beta barely matters (12..96: within 0.5 %)
constexpr int64_t kAlpha = 20, kBeta = 24;

}  // namespace

struct g5_bfs {
    g5_graph *g = nullptr;
    hipStream_t s = nullptr;
    int64_t wr = 0, wc = 0;  // row / column bitmap words
    uint64_t *d_visited = nullptr, *d_out = nullptr;
    uint32_t *d_parent = nullptr;
    int32_t *d_level = nullptr;
    int64_t alpha = kAlpha, beta = kBeta;  // direction switch of g5_bfs_run
    uint32_t *d_queue = nullptr;  // in-queue (local rows), sorted
    uint32_t *d_outq = nullptr;   // out-queue (local columns), sorted
    int64_t *d_qoff = nullptr;    // degree prefix over the in-queue, qlen + 1
    int64_t *d_scratch = nullptr;
    int64_t *d_cnt = nullptr;
    int64_t *h_cnt = nullptr;     // pinned mirror of d_cnt
    int64_t *d_part = nullptr;    // the workgroups' sums, 4 x kParts
    // the frontier's queue is in d_queue with its length in cnt[kQLen]; its
    // degree prefix in d_qoff with the total in cnt[kEdges].  Without a queue
    // the frontier is in d_inbits
    bool queue_ok = false, qoff_ok = false;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    g5::S4Codec codec;
    uint32_t *d_words = nullptr;  // codec stream for G5_RUN_CODEC
    size_t words_cap = 0;
    int64_t root = -1;
    int depth = -1;
    int64_t qlen = 0;
    // per-kernel accounting of k_expand (g5_bfs_profile / g5_bfs_stats)
    bool prof = false;
    hipEvent_t ek0 = nullptr, ek1 = nullptr;
    double exp_ms = 0, exp_bytes = 0;
    int64_t exp_launches = 0, exp_edges = 0;
    // bottom-up levels of g5_bfs_run: the next-frontier bitmap and accounting
    uint64_t *d_next = nullptr;
    double bu_ms = 0, bu_bytes = 0;
    int64_t bu_launches = 0, bu_edges = 0;
    // g5_bfs_run: vertices without edges (a diagonal block), visited from
    // the start so that no bottom-up level reads their offsets
    uint64_t *d_isolated = nullptr;
    // hook path: the row frontier as a bitmap (g5_bfs_set_in_bitmap), for
    // g5_bfs_expand_bottom_up
    uint64_t *d_inbits = nullptr;
    bool inbits_valid = false;
    // g5_bfs_run's levels on the device (k_level): a third frontier bitmap,
    // the two levels' queues and their prefixes (kGroups times gcap entries
    // each) and the control record.  6 bytes a vertex: allocated with the handle
    // of a whole graph, at the first g5_bfs_run of a grid's block, whose hooks
    // do without (level_buffers)
    uint64_t *d_third = nullptr;
    uint32_t *d_gq[2] = {nullptr, nullptr};
    int64_t *d_goff[2] = {nullptr, nullptr};
    int64_t gcap = 0;
    struct LevelCtl *d_ctl = nullptr;
};

namespace {

__device__ __forceinline__ int64_t src_of(const int64_t *__restrict__ qoff, int64_t lo, int64_t hi,
                                          int64_t e)
{
    // last s in [lo, hi] with qoff[s] <= e
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (qoff[mid] <= e) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// A queue given by the host: its degrees (for the prefix), its length, and the
// out-bitmap cleared for the expansion.
__global__ __launch_bounds__(256) void k_queue_degrees(const uint32_t *__restrict__ q, int64_t n,
                                                       const int64_t *__restrict__ rowptr,
                                                       int64_t *__restrict__ qoff, int64_t *__restrict__ cnt,
                                                       uint64_t *__restrict__ out, int64_t wc)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = t; i < n; i += stride) {
        const uint32_t u = q[i];
        qoff[i] = rowptr[u + 1] - rowptr[u];
    }
    for (int64_t w = t; w < wc; w += stride) out[w] = 0;
    if (t == 0) cnt[kQLen] = n;
}

// The sources of the edges [t0, t1) of a queue with its degree prefix: the
// first and the last by two waves' searches, all of them staged in LDS if they
// are few (two edges and more each on average).  All 256 threads call it.
struct TileSrc {
    int64_t lo, hi;
    bool staged;
};
__device__ __forceinline__ TileSrc stage_sources(const uint32_t *__restrict__ q, const int64_t *__restrict__ qoff,
                                                 int64_t qn, const int64_t *__restrict__ rowptr, int64_t t0,
                                                 int64_t t1, int64_t *s_range, int32_t *s_off, uint32_t *s_u,
                                                 int64_t *s_rb)
{
    if (threadIdx.x < 128) {
        const int64_t r = g5_wave_src_of(qoff, 0, qn - 1, threadIdx.x < 64 ? t0 : t1 - 1);
        if ((threadIdx.x & 63) == 0) s_range[threadIdx.x >> 6] = r;
    }
    __syncthreads();
    TileSrc t;
    t.lo = s_range[0];
    t.hi = s_range[1];
    t.staged = t.hi - t.lo < kTileSrc;
    if (t.staged)
        for (int j = threadIdx.x; j <= (int)(t.hi - t.lo); j += 256) {
            const uint32_t u = q[t.lo + j];
            const int64_t o = qoff[t.lo + j];
            s_u[j] = u;
            s_rb[j] = rowptr[u] - o;
            s_off[j] = (int32_t)max(o - t0, (int64_t)-1);
        }
    __syncthreads();
    return t;
}
// the source of edge e, and the edge's place in the columns
__device__ __forceinline__ uint32_t edge_source(const TileSrc &t, const uint32_t *__restrict__ q,
                                                const int64_t *__restrict__ qoff,
                                                const int64_t *__restrict__ rowptr, int64_t t0, int64_t e,
                                                const int32_t *s_off, const uint32_t *s_u, const int64_t *s_rb,
                                                int64_t &at)
{
    if (t.staged) {
        const int32_t rel = (int32_t)(e - t0);
        int x = 0, y = (int)(t.hi - t.lo);  // last source that starts at or before rel
        while (x < y) {
            const int mid = (x + y + 1) >> 1;
            if (s_off[mid] <= rel) x = mid;
            else y = mid - 1;
        }
        at = s_rb[x] + e;
        return s_u[x];
    }
    const int64_t x = src_of(qoff, t.lo, t.hi, e);
    const uint32_t u = q[x];
    at = rowptr[u] + (e - qoff[x]);
    return u;
}

// Top-down: the frontier's edges in tiles.  kCount: part[workgroup] = the out
// bits it was the first to set.  A search's top-down levels at scale 22 take 9
// us each (17 with one thread's search for a tile's first and last source and
// a search of the prefix in memory for every edge).
template <bool kCount>
__global__ __launch_bounds__(kExpandBlock) void k_expand(
    const uint32_t *__restrict__ q, const int64_t *__restrict__ qoff, const int64_t *__restrict__ cnt,
    const int64_t *__restrict__ rowptr, const uint32_t *__restrict__ cols,
    const uint64_t *__restrict__ visited, uint64_t *out, uint32_t *parent, int64_t *__restrict__ part)
{
    __shared__ int64_t s_range[2], s_rb[kTileSrc];
    __shared__ int32_t s_off[kTileSrc];
    __shared__ uint32_t s_u[kTileSrc];
    const int64_t qn = cnt[kQLen];
    const int64_t E = cnt[kEdges];
    int64_t found = 0;
    for (int64_t t0 = blockIdx.x * (int64_t)kExpandTile; t0 < E; t0 += (int64_t)gridDim.x * kExpandTile) {
        const int64_t t1 = min(E, t0 + (int64_t)kExpandTile);
        const TileSrc src = stage_sources(q, qoff, qn, rowptr, t0, t1, s_range, s_off, s_u, s_rb);
        // a thread's edges together, so that their loads are in flight at once
        constexpr int U = kExpandTile / kExpandBlock;
        uint32_t u[U], v[U];
        uint64_t seen[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int64_t e = t0 + threadIdx.x + k * kExpandBlock;
            u[k] = v[k] = kNoParent;
            if (e >= t1) continue;
            int64_t at;
            u[k] = edge_source(src, q, qoff, rowptr, t0, e, s_off, s_u, s_rb, at);
            v[k] = cols[at];
        }
#pragma unroll
        for (int k = 0; k < U; ++k) seen[k] = v[k] == kNoParent ? ~0ull : visited[v[k] >> 6];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int64_t w = v[k] >> 6;
            const uint64_t bit = 1ull << (v[k] & 63);
            if (seen[k] & bit) continue;
            if (!(out[w] & bit)) {
                if (kCount)
                    found += !(atomicOr((unsigned long long *)&out[w], (unsigned long long)bit) & bit);
                else
                    atomicOr((unsigned long long *)&out[w], (unsigned long long)bit);
            }
            if (parent[v[k]] > u[k]) atomicMin(&parent[v[k]], u[k]);
        }
        __syncthreads();
    }
    if (kCount) {
        found = g5_block_sum256(found);
        if (threadIdx.x == 0) part[blockIdx.x] = found;
    }
}

// visited |= in, out := the bits of in that are new, level := depth for them;
// part (if not null): a bitmap tile's new vertices, and with rowptr (1x1
// block) their degrees kTiles further.  in may be out.  A workgroup takes 64
// words at a time, 16 to a wave (lane j commits word w0 + j); then the wave
// walks the words with new bits 8 at a time, lane i taking vertex 64 w + i, so
// a word's level stores and offset reads are coalesced, and the 8 words'
// offset loads are all issued before any is used (a vertex's degree is the
// next lane's offset minus its own; lane 63 loads the next word's first
// offset).  The sums are stored per tile: added up with atomics on one
// address they took their turns (10 us a level at scale 22, now 5).
constexpr int kCommitGroup = 8;
constexpr int kCommitWords = 16;

__global__ __launch_bounds__(256) void k_commit(const uint64_t *in, uint64_t *out, uint64_t *__restrict__ visited,
                                                int32_t *__restrict__ level, int64_t wc, int64_t tile, int32_t depth,
                                                const int64_t *__restrict__ rowptr, int64_t *__restrict__ part)
{
    const int lane = __lane_id();
    const int64_t end = min(wc, (blockIdx.x + 1) * tile);
    int64_t c = 0, ce = 0;
    for (int64_t w0 = blockIdx.x * tile + (threadIdx.x >> 6) * kCommitWords; w0 < end; w0 += 64) {
        const int64_t w = w0 + lane;
        uint64_t nw = 0;
        if (lane < kCommitWords && w < end) {
            const uint64_t o = in[w];
            if (o) {
                const uint64_t vis = visited[w];
                nw = o & ~vis;
                if (nw) visited[w] = vis | nw;
                c += __popcll(nw);
            }
            if (nw != o || in != out) out[w] = nw;
        }
        const uint64_t todo = __ballot(nw != 0);
#pragma unroll
        for (int j0 = 0; j0 < kCommitWords; j0 += kCommitGroup) {
            if (((todo >> j0) & ((1ull << kCommitGroup) - 1)) == 0) continue;
            uint64_t bits[kCommitGroup];
            int64_t lo[kCommitGroup], hi[kCommitGroup];
#pragma unroll
            for (int k = 0; k < kCommitGroup; ++k) {
                bits[k] = g5_bcast64(nw, j0 + k);  // zero for words past the tile
                const int64_t v = (w0 + j0 + k) * 64 + lane;
                const bool any = bits[k] != 0;  // wave-uniform
                lo[k] = (rowptr && any) ? rowptr[v] : 0;
                hi[k] = (rowptr && any && lane == 63) ? rowptr[v + 1] : 0;
                if (bits[k] >> lane & 1) level[v] = depth;
            }
#pragma unroll
            for (int k = 0; k < kCommitGroup; ++k) {
                const int64_t nxt = __shfl_down(lo[k], 1, 64);
                const int64_t up = lane == 63 ? hi[k] : nxt;
                if (bits[k] >> lane & 1) ce += up - lo[k];
            }
        }
    }
    if (!part) return;
    c = g5_block_sum256(c);
    ce = g5_block_sum256(ce);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = c;
        part[g5::kTiles + blockIdx.x] = ce;
    }
}

// Bottom-up scans: every unvisited vertex looks through its neighbours in
// ascending id order for the first one whose frontier bit is set -- its
// minimum-id frontier neighbour, the parent CPUBFS_bin's ascending scan keeps
// (cpu_2d/cpubfs_bin.cpp:150-173).  One wavefront per 64-vertex bitmap word
// (lane = vertex), so the next-frontier word is the wave's ballot and needs no
// atomics.
//
// A lane looks at its own row's first kBuFirst neighbours, where a dense
// level's scans end.  The rows still open then share the wave: r of them get
// 64 / r lanes each (a power of two), which take that many consecutive
// neighbours kBuSteps times over, until all rows have ended.  A lane alone on a
// long row is a chain of dependent loads with the other lanes idle, and its
// row's lines are gone from the caches before the next step reads on.
// Measured over a search's three bottom-up levels, commit included: 143 us at
// scale 22 (lane per row to its end: 455), 500 at 24, 3.2 ms at 26 (3.5).
// The first level's random frontier bits bound it, about one address per
// clock and CU, then the row starts' lines.  kBuFirst 2 and 4: 1.02 and 1.13
// times that at scale 24; kBuSteps 2: 1.07.
constexpr int kBuFirst = 1;
constexpr int kBuSteps = 1;
struct BuScan {  // one wave's
    int64_t at[64], end[64];
    uint32_t owner[64], par[64];
};

__device__ __forceinline__ void bu_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The first frontier neighbour in [j, e) of each lane's row (none: kNoParent;
// j == e for lanes without a row); j becomes the end of what was looked at.
__device__ __forceinline__ uint32_t bu_scan(int64_t &j, int64_t e, const uint32_t *__restrict__ cols,
                                            const uint64_t *__restrict__ front, BuScan &s, int lane)
{
    uint32_t par = kNoParent;
    {
        uint32_t u[kBuFirst];
        uint64_t fw[kBuFirst];
#pragma unroll
        for (int k = 0; k < kBuFirst; ++k) u[k] = j + k < e ? cols[j + k] : 0u;
#pragma unroll
        for (int k = 0; k < kBuFirst; ++k) fw[k] = j + k < e ? front[u[k] >> 6] : 0ull;
#pragma unroll
        for (int k = kBuFirst - 1; k >= 0; --k)
            if (fw[k] >> (u[k] & 63) & 1) par = u[k];
        j = min(e, j + kBuFirst);
    }
    uint64_t open = __ballot(par == kNoParent && j < e);
    while (open) {
        const int r = __popcll(open);
        const int lg = r > 1 ? 6 - (32 - __clz(r - 1)) : 6;  // log2 of the lanes per row
        const bool mine = open >> lane & 1;
        if (mine) {
            const int rank = __popcll(open & ((1ull << lane) - 1));
            s.at[rank] = j;
            s.end[rank] = e;
            s.owner[rank] = lane;
            s.par[lane] = kNoParent;
        }
        bu_wave_sync();
        const int row = lane >> lg;
        int64_t at = 0, end = 0;
        uint32_t owner = 0;
        if (row < r) {
            at = s.at[row] + (lane & ((1 << lg) - 1));
            end = s.end[row];
            owner = s.owner[row];
        }
        uint32_t u[kBuSteps];
        uint64_t fw[kBuSteps];
#pragma unroll
        for (int k = 0; k < kBuSteps; ++k) u[k] = at + (k << lg) < end ? cols[at + (k << lg)] : 0u;
#pragma unroll
        for (int k = 0; k < kBuSteps; ++k) fw[k] = at + (k << lg) < end ? front[u[k] >> 6] : 0ull;
        // the row's first hit: the lowest lane of the earliest step
        const uint64_t below = ((1ull << lane) - 1) & ~((1ull << (row << lg)) - 1);
        const uint64_t group = lg == 6 ? ~0ull : ((1ull << (1 << lg)) - 1) << ((row << lg) & 63);
        bool over = false;  // an earlier step hit
#pragma unroll
        for (int k = 0; k < kBuSteps; ++k) {
            const bool hit = fw[k] >> (u[k] & 63) & 1;
            const uint64_t hits = __ballot(hit);
            if (hit && !over && !(hits & below)) s.par[owner] = u[k];
            over = over || (hits & group);
        }
        bu_wave_sync();
        if (mine) {
            par = s.par[lane];
            j = min(e, j + (kBuSteps << lg));
        }
        open = __ballot(mine && par == kNoParent && j < e);
    }
    return par;
}

// kCommit: with the level's commit (visited, levels) in the same pass.
// part[j * kParts + workgroup]: new vertices, their degrees (with the row
// offsets of their own rows), neighbours checked, vertices scanned.  Three
// atomics per workgroup on one line were most of its time before: at scale 22,
// commit included, a level (of three) took 149 us, now 36.
enum BuPart { kPNew = 0, kPNewEdges = 1, kPBuEdges = 2, kPBuVerts = 3 };

template <bool kCommit>
__global__ __launch_bounds__(256) void k_bottom_up(const int64_t *__restrict__ rowptr,
                                                   const uint32_t *__restrict__ cols,
                                                   uint64_t *__restrict__ visited,
                                                   const uint64_t *__restrict__ front, uint64_t *__restrict__ next,
                                                   uint32_t *__restrict__ parent, int32_t *__restrict__ level,
                                                   int32_t depth, int64_t wc, int64_t *__restrict__ part)
{
    __shared__ BuScan s_scan[4];
    const int lane = __lane_id();
    int64_t nedges = 0, nverts = 0, newdeg = 0, nnew = 0;
    for (int64_t w = blockIdx.x * 4 + (threadIdx.x >> 6); w < wc; w += (int64_t)gridDim.x * 4) {
        const uint64_t vis = visited[w];
        const int64_t v = w * 64 + lane;
        int64_t b = 0, e = 0;
        if (!(vis >> lane & 1)) {
            b = rowptr[v];
            e = rowptr[v + 1];
            ++nverts;
        }
        int64_t j = b;
        const uint32_t par = bu_scan(j, e, cols, front, s_scan[threadIdx.x >> 6], lane);
        const bool hit = par != kNoParent;
        if (hit) {
            parent[v] = par;
            if (kCommit) level[v] = depth;
            newdeg += e - b;
            ++nnew;
        }
        nedges += j - b;
        const uint64_t bits = __ballot(hit);
        if (lane == 0) {
            next[w] = bits;
            if (kCommit && bits) visited[w] = vis | bits;
        }
    }
    nnew = g5_block_sum256(nnew);
    newdeg = g5_block_sum256(newdeg);
    nedges = g5_block_sum256(nedges);
    nverts = g5_block_sum256(nverts);
    if (threadIdx.x == 0) {
        part[kPNew * kParts + blockIdx.x] = nnew;
        part[kPNewEdges * kParts + blockIdx.x] = newdeg;
        part[kPBuEdges * kParts + blockIdx.x] = nedges;
        part[kPBuVerts * kParts + blockIdx.x] = nverts;
    }
}

// A search's state at its start, in one launch (a fill each took seven): the
// root's column visited at level 0 (isolated: with the edgeless vertices), its
// bit in out (the frontier of a bottom-up first level), its row the queue.
// n_cols is a multiple of 64.
__global__ __launch_bounds__(256) void k_start(int64_t root_row, int64_t root_col, int64_t wc, int64_t n_cols,
                                               const uint64_t *__restrict__ isolated,
                                               const int64_t *__restrict__ rowptr, uint64_t *__restrict__ visited,
                                               uint64_t *__restrict__ out, uint64_t *__restrict__ next,
                                               uint32_t *__restrict__ parent, int32_t *__restrict__ level,
                                               uint32_t *__restrict__ queue, int64_t *__restrict__ qoff,
                                               int64_t *__restrict__ cnt)
{
    const int64_t t = blockIdx.x * 256ll + threadIdx.x, stride = gridDim.x * 256ll;
    for (int64_t w = t; w < wc; w += stride) {
        const uint64_t bit = root_col >= 0 && w == root_col >> 6 ? 1ull << (root_col & 63) : 0ull;
        visited[w] = (isolated ? isolated[w] : 0ull) | bit;
        out[w] = bit;
        next[w] = 0;
    }
    uint4 *p4 = (uint4 *)parent, *l4 = (uint4 *)level;
    for (int64_t i = t; i < n_cols / 4; i += stride) {
        const int at = i == root_col >> 2 ? (int)(root_col & 3) : 4;  // root_col -1: never
        p4[i] = make_uint4(at == 0 ? kRootMark : kNoParent, at == 1 ? kRootMark : kNoParent,
                           at == 2 ? kRootMark : kNoParent, at == 3 ? kRootMark : kNoParent);
        l4[i] = make_uint4(at == 0 ? 0u : ~0u, at == 1 ? 0u : ~0u, at == 2 ? 0u : ~0u, at == 3 ? 0u : ~0u);
    }
    if (t < kNCnt) {
        int64_t c = 0;
        if (root_row >= 0 && t == kQLen) {
            c = 1;
            queue[0] = (uint32_t)root_row;
            qoff[0] = 0;
        }
        if (root_row >= 0 && t == kEdges) c = rowptr[root_row + 1] - rowptr[root_row];
        cnt[t] = c;
    }
}

__global__ __launch_bounds__(256) void k_copy_words(const uint64_t *__restrict__ from, uint64_t *__restrict__ to,
                                                    int64_t n)
{
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) to[i] = from[i];
}

__global__ void k_result(const uint32_t *__restrict__ parent, int64_t n, int64_t row_start,
                         int64_t col_start, int64_t *__restrict__ pred)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t p = parent[i];
        pred[i] = p == kNoParent ? -1 : (p == kRootMark ? i + col_start : (int64_t)p + row_start);
    }
}

constexpr int kSumGrid = 2048;

// part[workgroup] = its share of the sum (one atomic each on one address, 1024
// of them, were 4 us); n is a multiple of 64
__global__ __launch_bounds__(256) void k_nedge(const uint32_t *__restrict__ gdeg, const int32_t *__restrict__ level,
                                               int64_t n, int64_t *__restrict__ part)
{
    const uint4 *g4 = (const uint4 *)gdeg;
    const int4 *l4 = (const int4 *)level;
    int64_t c = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n / 4;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int4 l = l4[i];
        const uint4 g = g4[i];
        c += (int64_t)(l.x >= 0 ? g.x : 0u) + (l.y >= 0 ? g.y : 0u) + (int64_t)(l.z >= 0 ? g.z : 0u) +
             (l.w >= 0 ? g.w : 0u);
    }
    c = g5_block_sum256(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

// nedge's generated-degree sum and the predecessor-map checksum of a 1x1
// search in one pass: sum over reached v of mix64(v << 32 | (pred(v) + 1))
__global__ void k_summary(const uint32_t *__restrict__ gdeg, const int32_t *__restrict__ level,
                          const uint32_t *__restrict__ parent, int64_t n, int64_t *__restrict__ part)
{
    int64_t c = 0;
    uint64_t h = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        if (level[i] >= 0) {
            c += gdeg[i];
            const uint32_t p = parent[i];
            const uint64_t pred = p == kRootMark ? (uint64_t)i : (uint64_t)p;
            h += g5_mix64(((uint64_t)i << 32) | (uint32_t)(pred + 1));
        }
    c = g5_block_sum256(c);
    h = g5_block_sum256_u64(h);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = c;
        part[kParts + blockIdx.x] = (int64_t)h;
    }
}

// The frontier of d_inbits or of a host's queue as a queue with its degree
// prefix, and out cleared: one to three launches before an expansion, none of
// them where the level before left both.
int prepare_queue(g5_bfs *b, uint64_t *out)
{
    g5_graph *g = b->g;
    hipStream_t s = b->s;
    if (b->queue_ok && b->qoff_ok) {
        G5_HIP(g5::fill_u64(out, b->wc, 0, s));
    } else if (b->queue_ok) {
        hipLaunchKernelGGL(k_queue_degrees, g5::grid_for(std::max(b->qlen, b->wc), 256, 4096), 256, 0, s,
                           (const uint32_t *)b->d_queue, b->qlen, (const int64_t *)g->d_rowptr, b->d_qoff, b->d_cnt,
                           out, b->wc);
        G5_HIP(hipGetLastError());
        G5_HIP(g5::exclusive_scan_i64(b->d_qoff, b->qlen, b->d_cnt + kEdges, b->d_scratch, s));
    } else {
        g5::QueueOut o{};
        o.q = b->d_queue;
        o.qoff = b->d_qoff;
        o.d_n = b->d_cnt + kQLen;
        o.d_e = b->d_cnt + kEdges;
        o.clear = out;
        o.n_clear = b->wc;
        G5_HIP(g5::bitmap_to_queue(b->d_inbits, b->wr, (const int64_t *)g->d_rowptr, o, b->d_part, false, s));
    }
    b->queue_ok = b->qoff_ok = true;
    return G5_OK;
}

// One level's expansion from the queue (d_queue, d_qoff, cnt[kQLen] and
// cnt[kEdges]) into out; count: part[0 .. kExpandGrid) sum to its new bits.
// E: its edges if the host knows them, else -1.
int expand_level(g5_bfs *b, uint64_t *out, bool count, int64_t E)
{
    g5_graph *g = b->g;
    hipStream_t s = b->s;
    if (b->prof) G5_HIP(hipEventRecord(b->ek0, s));
    static_assert(kExpandGrid <= kParts, "a sum per workgroup");
    hipLaunchKernelGGL(count ? k_expand<true> : k_expand<false>,
                       count || E < 0 ? kExpandGrid : g5::grid_for(E, kExpandTile, kExpandGrid), kExpandBlock, 0, s,
                       (const uint32_t *)b->d_queue, (const int64_t *)b->d_qoff, (const int64_t *)b->d_cnt,
                       (const int64_t *)g->d_rowptr, (const uint32_t *)g->d_cols, (const uint64_t *)b->d_visited, out,
                       b->d_parent, b->d_part);
    G5_HIP(hipGetLastError());
    if (b->prof) G5_HIP(hipEventRecord(b->ek1, s));
    return G5_OK;
}

// The workgroups' n sums in d_part (arrays stride apart, the first k of
// them) to the counters slot[0 .. k) in pinned memory, and the codec's error
// flag with them.  frontier: the first two are also the next frontier's
// vertices and edges.  Waits for the stream.
int fold_counters(g5_bfs *b, int64_t stride, int n, const int *slot, int k, bool frontier)
{
    g5::FoldOut o{};
    for (int j = 0; j < k; ++j) o.host[j] = b->h_cnt + slot[j];
    if (frontier) {
        o.dev[0] = b->d_cnt + kQLen;
        o.dev[1] = b->d_cnt + kEdges;
    }
    o.from = b->d_cnt + kCodecErr;
    o.to = b->h_cnt + kCodecErr;
    o.ncopy = 1;
    G5_HIP(g5::fold_parts(b->d_part, stride, n, o, b->s));
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

// After the level's counters are on the host: k_expand time and its
// algorithmic bytes, 16 B row-offset pair per frontier vertex, 4 B column id
// + 8 B visited word per frontier edge, 8 B out word + 4 B parent per newly
// reached vertex.
int account_level(g5_bfs *b, int64_t qlen, int64_t E, int64_t n_new)
{
    if (!b->prof || qlen == 0) return G5_OK;
    float ms = 0;
    G5_HIP(hipEventElapsedTime(&ms, b->ek0, b->ek1));
    b->exp_ms += ms;
    b->exp_launches += 1;
    b->exp_edges += E;
    b->exp_bytes += 16.0 * qlen + 12.0 * E + 12.0 * n_new;
    return G5_OK;
}

// After a bottom-up level: k_bottom_up time and its algorithmic bytes, 16 B
// row-offset pair per unvisited vertex scanned, 4 B column + 8 B frontier
// word per neighbour checked, 4 B parent per newly reached vertex, 16 B
// (visited read + next write) per 64-vertex word; with the commit in the same
// pass 4 B level per new vertex and 8 B visited per word more.
int account_bottom_up(g5_bfs *b, int64_t n_new, bool commit)
{
    if (!b->prof) return G5_OK;
    float ms = 0;
    G5_HIP(hipEventElapsedTime(&ms, b->ek0, b->ek1));
    const int64_t E = b->h_cnt[kBuEdges], V = b->h_cnt[kBuVerts];
    b->bu_ms += ms;
    b->bu_launches += 1;
    b->bu_edges += E;
    b->bu_bytes += 16.0 * V + 12.0 * E + (commit ? 8.0 : 4.0) * n_new + (commit ? 24.0 : 16.0) * b->wc;
    return G5_OK;
}

// bit v of word v / 64: row v of the (diagonal) block has no neighbours
__global__ void k_isolated(const int64_t *__restrict__ rowptr, int64_t wc, uint64_t *__restrict__ bits)
{
    const int lane = __lane_id();
    for (int64_t w = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6; w < wc;
         w += ((int64_t)gridDim.x * blockDim.x) >> 6) {
        const int64_t v = w * 64 + lane;
        const uint64_t word = __ballot(rowptr[v + 1] == rowptr[v]);
        if (lane == 0) bits[w] = word;
    }
}

// d_isolated, at the first search of a resident graph
int find_isolated(g5_bfs *b)
{
    if (b->d_isolated) return G5_OK;
    G5_HIP(hipMalloc(&b->d_isolated, (size_t)(b->wc ? b->wc : 1) * 8));
    hipLaunchKernelGGL(k_isolated, g5::grid_for(b->wc * 64, 256, 4096), 256, 0, b->s,
                       (const int64_t *)b->g->d_rowptr, b->wc, b->d_isolated);
    G5_HIP(hipGetLastError());
    return G5_OK;
}

// isolated: start with the block's edgeless vertices visited (g5_bfs_run on a
// diagonal block: they are never reached, so results do not change)
int reset_search(g5_bfs *b, int64_t root, bool isolated = false)
{
    g5_graph *g = b->g;
    hipStream_t s = b->s;
    const int64_t rr = root - g->row_start, rc = root - g->col_start;
    const int64_t root_row = (root >= 0 && rr >= 0 && rr < g->n_rows) ? rr : -1;
    const int64_t root_col = (root >= 0 && rc >= 0 && rc < g->n_cols) ? rc : -1;
    hipLaunchKernelGGL(k_start, g5::grid_for(g->n_cols / 4, 256, 4096), 256, 0, s, root_row, root_col, b->wc,
                       g->n_cols, isolated ? (const uint64_t *)b->d_isolated : (const uint64_t *)nullptr,
                       (const int64_t *)g->d_rowptr, b->d_visited, b->d_out, b->d_next, b->d_parent, b->d_level,
                       b->d_queue, b->d_qoff, b->d_cnt);
    G5_HIP(hipGetLastError());
    b->root = root;
    b->depth = 0;
    b->qlen = root_row >= 0 ? 1 : 0;
    b->queue_ok = b->qoff_ok = true;
    b->inbits_valid = false;
    return G5_OK;
}

// ---- the resident search, decided on the device ----
//
// g5_bfs_run's levels as one kernel each, with no word from the host between
// them: every workgroup reads the level before's totals, takes the same
// decision (done, top-down or bottom-up), and does its share.  A level costs
// one launch (about 10 before, and a host round trip); the host looks only
// after a batch of levels.  A whole search with its maps and count: 399 -> 133
// us at scale 16, 3.9-4.3 -> 3.3-3.6 ms at 26.
//
// Three frontier bitmaps rotate: a level reads the frontier, writes the next
// one and clears the third.  Visited lags one level behind: the frontier is
// merged into it by the level that expands it, so "visited" below is always
// visited | frontier.  Both directions collect the new vertices per workgroup
// in LDS and append them, with their degree prefix, to one of the next level's
// kGroups queues; one packed atomic (vertices, edges) reserves both and is the
// queue's total.  (Returning atomics on one address take 12 ns each: 100 us of
// a level whose 8192 workgroups all append to one queue.)  The queues
// are in no order, which no result depends on.  They are only complete
// if the next level may run top-down: a workgroup whose buffer overflows (a
// dense bottom-up level), a full queue, or a top-down level that has already
// found more edges than the switch allows leave it out, and the next level
// runs bottom-up.  From then on the level's totals need not be exact (the next
// level's direction is settled, and some vertex was found), so workgroups that
// see it collect nothing any more.
constexpr int kLvBlock = 256;
constexpr int kLvGrid = 4096;   // two rounds of 8 workgroups per CU, which differ in what they take
constexpr int kLvTile = 1024;   // edges of a top-down tile
constexpr int kLvBuf = 1024;    // new vertices a workgroup keeps
constexpr int kLvMem = 4096;    // words of LDS: the buffer and staged sources, or the scans' rows
constexpr int kEdgeBits = 34;   // of a packed total; the vertices take the rest
constexpr uint64_t kEdgeMask = (1ull << kEdgeBits) - 1;
constexpr int kGroups = 16;
constexpr int kMinQueue = 4096;  // entries of a group's queue at least

enum Mode { kTopDown = 0, kBottomUp = 1, kDone = 2 };

}  // namespace

struct LevelCtl {
    // written by level d at [d % 2], read by level d + 1
    struct {
        int64_t mode, m_u;
    } lv[2];
    int64_t pad[12];
    // level d at [d % 3], every word in a line of its own: the groups' packed
    // new vertices and edges, and whether the queues are incomplete (a hint
    // within the level, so it is read and written through the XCD's own L2)
    struct {
        unsigned long long x;
        unsigned long long pad[15];
    } tot[3][16], lost[3];
};

namespace {

struct LevelArgs {
    const int64_t *rowptr;
    const uint32_t *cols;
    uint64_t *visited;
    uint32_t *parent;
    int32_t *level;
    // this level's frontier, the next one's, and the bitmap to clear; its
    // queue and prefix, and the next one's.  The host picks them (an index
    // into arrays here would make every access to them a flat one)
    uint64_t *front, *next, *third;
    uint32_t *q, *qn;
    int64_t *qoff, *qoffn;
    LevelCtl *ctl;
    int64_t *host;
    int64_t n, wc, nnz, alpha, beta;
    int64_t gcap;  // entries of a group's queue
};

// what a level's workgroups know of the frontier's queues
struct Groups {
    int64_t n[kGroups], edges[kGroups], tile0[kGroups + 1];
};

// The search's state at its start: visited = the edgeless vertices, the root
// the only frontier vertex; one kernel.
__global__ __launch_bounds__(kLvBlock) void k_reset(LevelArgs a, const uint64_t *__restrict__ isolated, int64_t root)
{
    const int64_t t = blockIdx.x * (int64_t)kLvBlock + threadIdx.x, stride = (int64_t)gridDim.x * kLvBlock;
    for (int64_t w = t; w < a.wc; w += stride) {
        a.visited[w] = isolated[w];
        a.front[w] = w == root >> 6 ? 1ull << (root & 63) : 0ull;
        a.next[w] = 0;
        a.third[w] = 0;
    }
    // n is a multiple of 64
    uint4 *p4 = (uint4 *)a.parent, *l4 = (uint4 *)a.level;
    for (int64_t i = t; i < a.n / 4; i += stride) {
        const int at = i == root >> 2 ? (int)(root & 3) : 4;
        p4[i] = make_uint4(at == 0 ? kRootMark : kNoParent, at == 1 ? kRootMark : kNoParent,
                           at == 2 ? kRootMark : kNoParent, at == 3 ? kRootMark : kNoParent);
        l4[i] = make_uint4(at == 0 ? 0u : ~0u, at == 1 ? 0u : ~0u, at == 2 ? 0u : ~0u, at == 3 ? 0u : ~0u);
    }
    if (blockIdx.x == 0) {
        for (int i = threadIdx.x; i < (int)(sizeof(LevelCtl) / 8); i += kLvBlock) ((uint64_t *)a.ctl)[i] = 0;
        __syncthreads();
        if (threadIdx.x == 0) {
            static_assert(kGroups <= 16, "totals");
            a.q[0] = (uint32_t)root;
            a.qoff[0] = 0;
            a.ctl->lv[1].mode = kTopDown;
            a.ctl->lv[1].m_u = a.nnz;
            a.ctl->tot[2][0].x = 1ull << kEdgeBits | (unsigned long long)(a.rowptr[root + 1] - a.rowptr[root]);
        }
    }
}

// whether the level's queue is known to be incomplete
__device__ __forceinline__ bool lost_yet(const LevelArgs &a, int d)
{
    return __hip_atomic_load(&a.ctl->lost[d % 3].x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0;
}
__device__ __forceinline__ void set_lost(const LevelArgs &a, int d)
{
    __hip_atomic_store(&a.ctl->lost[d % 3].x, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The workgroup's new vertices s_v[0 .. cnt) of degrees s_d go to the queue
// (all threads call it, after a barrier; s_v is free again after the next one)
__device__ __forceinline__ void level_flush(const LevelArgs &a, int d, int64_t limit, int cnt, const uint32_t *s_v,
                                            const uint32_t *s_d)
{
    __shared__ int64_t s_wave[kLvBlock / 64];
    __shared__ unsigned long long s_at;
    const int per = (cnt + kLvBlock - 1) / kLvBlock, i0 = threadIdx.x * per, i1 = min(cnt, i0 + per);
    int64_t sum = 0;
    for (int i = i0; i < i1; ++i) sum += s_d[i];
    const int64_t inc = g5_wave_incl_scan(sum);
    if ((threadIdx.x & 63) == 63) s_wave[threadIdx.x >> 6] = inc;
    __syncthreads();
    int64_t before = inc - sum, all = 0;
    for (int w = 0; w < kLvBlock / 64; ++w) {
        before += w < (int)(threadIdx.x >> 6) ? s_wave[w] : 0;
        all += s_wave[w];
    }
    if (threadIdx.x == 0)
        s_at = atomicAdd(&a.ctl->tot[d % 3][blockIdx.x % kGroups].x,
                         (unsigned long long)cnt << kEdgeBits | (unsigned long long)all);
    __syncthreads();
    const int64_t pos = (int64_t)(s_at >> kEdgeBits), off = (int64_t)(s_at & kEdgeMask);
    if (pos + cnt <= a.gcap && off <= limit) {
        const int64_t base = (int64_t)(blockIdx.x % kGroups) * a.gcap + pos;
        int64_t run = off + before;
        for (int i = i0; i < i1; ++i) {
            a.qn[base + i] = s_v[i];
            a.qoffn[base + i] = run;
            run += s_d[i];
        }
    } else if (threadIdx.x == 0) {
        set_lost(a, d);
    }
}

// Top-down: the queue's edges in tiles, every tile's sources staged in LDS.
// The thread that sets a target's bit in the next frontier collects it; the
// parent is lowered to the smallest source with atomicMin.
__device__ __forceinline__ void level_top_down(const LevelArgs &a, int d, const Groups &gr, int64_t limit,
                                               uint32_t *s_mem)
{
    __shared__ int64_t s_range[2];
    __shared__ int s_n;
    __shared__ unsigned int s_lost;
    int32_t *s_off = (int32_t *)s_mem;                        // kTileSrc
    uint32_t *s_u = s_mem + kTileSrc;                           // kTileSrc
    int64_t *s_rb = (int64_t *)(s_mem + 2 * kTileSrc);          // kTileSrc
    uint32_t *s_v = s_mem + 4 * kTileSrc, *s_d = s_v + kLvBuf;  // kLvBuf each
    static_assert(4 * kTileSrc + 2 * kLvBuf <= kLvMem && kLvBuf >= kLvTile, "LDS");
    const uint64_t *__restrict__ front = a.front;
    if (threadIdx.x == 0) {
        s_n = 0;
        s_lost = 0;
    }
    for (int64_t w = blockIdx.x * (int64_t)kLvBlock + threadIdx.x; w < a.wc; w += (int64_t)gridDim.x * kLvBlock) {
        const uint64_t f = front[w];
        if (f) a.visited[w] |= f;
        a.third[w] = 0;
    }
    __syncthreads();
    for (int64_t t = blockIdx.x; t < gr.tile0[kGroups]; t += gridDim.x) {
        const int lane = threadIdx.x & 63;
        const int g = __popcll(__ballot(lane < kGroups && gr.tile0[lane] <= t)) - 1;  // the last such has tiles
        const uint32_t *__restrict__ q = a.q + g * a.gcap;
        const int64_t *__restrict__ qoff = a.qoff + g * a.gcap;
        const int64_t t0 = (t - gr.tile0[g]) * kLvTile, t1 = min(gr.edges[g], t0 + (int64_t)kLvTile);
        const int64_t qn = gr.n[g];
        if (threadIdx.x == 128) s_lost = lost_yet(a, d);
        const TileSrc src = stage_sources(q, qoff, qn, a.rowptr, t0, t1, s_range, s_off, s_u, s_rb);
        const bool collect = s_lost == 0;
        // a thread's edges together, so that their loads are in flight at once
        constexpr int U = kLvTile / kLvBlock;
        uint32_t u[U], v[U];
        uint64_t seen[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int64_t e = t0 + threadIdx.x + k * kLvBlock;
            u[k] = v[k] = kNoParent;
            if (e >= t1) continue;
            int64_t at;
            u[k] = edge_source(src, q, qoff, a.rowptr, t0, e, s_off, s_u, s_rb, at);
            v[k] = a.cols[at];
        }
#pragma unroll
        for (int k = 0; k < U; ++k) seen[k] = v[k] == kNoParent ? ~0ull : a.visited[v[k] >> 6];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int64_t w = v[k] >> 6;
            const uint64_t bit = 1ull << (v[k] & 63);
            if (seen[k] & bit) continue;
            if (front[w] & bit) continue;
            const bool early = !(a.next[w] & bit);
            if (early) {
                if (!collect) {
                    // the next level, bottom-up, writes the levels
                    atomicOr((unsigned long long *)&a.next[w], (unsigned long long)bit);
                } else if (!(atomicOr((unsigned long long *)&a.next[w], (unsigned long long)bit) & bit)) {
                    a.level[v[k]] = d + 1;
                    const int i = atomicAdd(&s_n, 1);
                    s_v[i] = v[k];
                    s_d[i] = (uint32_t)(a.rowptr[v[k] + 1] - a.rowptr[v[k]]);
                }
            }
            // an early source's parent slot holds nothing smaller yet
            if (early || a.parent[v[k]] > u[k]) atomicMin(&a.parent[v[k]], u[k]);
        }
        __syncthreads();
        const int cnt = s_n;
        if (cnt > kLvBuf - kLvTile) {
            level_flush(a, d, limit, cnt, s_v, s_d);
            __syncthreads();
            if (threadIdx.x == 0) s_n = 0;
            __syncthreads();
        }
    }
    const int cnt = s_n;
    if (cnt) level_flush(a, d, limit, cnt, s_v, s_d);
}

// Bottom-up: as k_bottom_up, a wave per 64-vertex word, with the level's
// commit (levels, visited, the next frontier) in the same pass.
__device__ __forceinline__ void level_bottom_up(const LevelArgs &a, int d, const int64_t *__restrict__ rowptr,
                                                const uint32_t *__restrict__ cols,
                                                const uint64_t *__restrict__ front, uint64_t *__restrict__ visited,
                                                uint64_t *__restrict__ next, uint64_t *__restrict__ third,
                                                uint32_t *__restrict__ parent, int32_t *__restrict__ level,
                                                bool late, uint32_t *s_mem)
{
    __shared__ int s_n;
    __shared__ unsigned int s_lost;
    constexpr int kCap = kLvBuf;
    uint32_t *s_v = s_mem, *s_d = s_mem + kCap;
    static_assert(2 * kCap * 4 + sizeof(BuScan) * (kLvBlock / 64) <= kLvMem * 4 && 2 * kCap * 4 % 16 == 0, "LDS");
    BuScan &s_scan = ((BuScan *)(s_mem + 2 * kCap))[threadIdx.x >> 6];
    const int lane = __lane_id();
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for (int64_t w = blockIdx.x * (int64_t)(kLvBlock / 64) + (threadIdx.x >> 6); w < a.wc;
         w += (int64_t)gridDim.x * (kLvBlock / 64)) {
        const uint64_t fr = front[w], vis = visited[w] | fr;
        const int64_t v = w * 64 + lane;
        if (late && (fr >> lane & 1)) level[v] = d;  // found by a top-down level that left them out
        int64_t b = 0, e = 0;
        if (!(vis >> lane & 1)) {
            b = rowptr[v];
            e = rowptr[v + 1];
        }
        const int64_t deg = e - b;
        const uint32_t par = bu_scan(b, e, cols, front, s_scan, lane);
        const bool hit = par != kNoParent;
        if (hit) {
            parent[v] = par;
            level[v] = d + 1;
        }
        const uint64_t bits = __ballot(hit);
        if (lane == 0) {
            next[w] = bits;
            visited[w] = vis | bits;
            third[w] = 0;
        }
        // the workgroup's new vertices, as long as they fit
        if (bits) {
            const int c = __popcll(bits);
            int i = 0;
            if (lane == 0) i = s_n <= kCap ? atomicAdd(&s_n, c) : kCap;
            i = __builtin_amdgcn_readfirstlane(i) + __popcll(bits & ((1ull << lane) - 1));
            if (hit && i < kCap) {
                s_v[i] = (uint32_t)v;
                s_d[i] = (uint32_t)deg;
            }
        }
    }
    if (threadIdx.x == 0) s_lost = lost_yet(a, d);
    __syncthreads();
    const int cnt = s_n;
    if (cnt == 0 || s_lost) return;
    if (cnt <= kCap) {
        level_flush(a, d, INT64_MAX, cnt, s_v, s_d);
    } else if (threadIdx.x == 0) {
        // some vertices (the next level only asks if there are any)
        atomicAdd(&a.ctl->tot[d % 3][blockIdx.x % kGroups].x, (unsigned long long)cnt << kEdgeBits);
        set_lost(a, d);
    }
}

__global__ __launch_bounds__(kLvBlock) void k_level(LevelArgs a, int d, const int64_t *__restrict__ rowptr,
                                                    const uint32_t *__restrict__ cols,
                                                    const uint64_t *__restrict__ front,
                                                    uint64_t *__restrict__ visited, uint64_t *__restrict__ next,
                                                    uint64_t *__restrict__ third, uint32_t *__restrict__ parent,
                                                    int32_t *__restrict__ level)
{
    __shared__ __align__(16) uint32_t s_mem[kLvMem];
    __shared__ int64_t s_mode, s_limit;
    __shared__ bool s_late;
    __shared__ Groups s_gr;
    if (a.ctl->lv[(d + 1) & 1].mode == kDone) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl->lv[d & 1].mode = kDone;
        return;
    }
    if (threadIdx.x < 64) {
        const int g = threadIdx.x;
        const unsigned long long tot = g < kGroups ? a.ctl->tot[(d + 2) % 3][g].x : 0ull;
        const int64_t n = (int64_t)(tot >> kEdgeBits), m = (int64_t)(tot & kEdgeMask);
        const int64_t tiles = (m + kLvTile - 1) / kLvTile, tinc = g5_wave_incl_scan(tiles);
        if (g < kGroups) {
            s_gr.n[g] = n;
            s_gr.edges[g] = m;
            s_gr.tile0[g] = tinc - tiles;
            if (g == kGroups - 1) s_gr.tile0[kGroups] = tinc;
        }
        const int64_t n_f = g5_wave_sum(n), m_f = g5_wave_sum(m);
        if (blockIdx.x == 0 && g < kGroups) a.ctl->tot[(d + 1) % 3][g].x = 0;
        if (g == 0) {
            const int64_t was = a.ctl->lv[(d + 1) & 1].mode;
            int64_t mode = was, m_u = a.ctl->lv[(d + 1) & 1].m_u;
            bool late = false;
            if (n_f == 0) mode = kDone;
            else if (d > 0) {  // the first level is top-down
                if (mode == kTopDown && m_f > m_u / a.alpha) mode = kBottomUp;
                else if (mode == kBottomUp && n_f < a.n / a.beta) mode = kTopDown;
                if (a.ctl->lost[(d + 2) % 3].x) mode = kBottomUp;
                late = mode == kBottomUp && was == kTopDown;
                if (mode == kTopDown) m_u -= m_f;
            }
            if (blockIdx.x == 0) {
                a.ctl->lv[d & 1].mode = mode;
                a.ctl->lv[d & 1].m_u = m_u;
                a.ctl->lost[(d + 1) % 3].x = 0;
                // the first level that finds its frontier empty says so
                if (mode == kDone) *a.host = d;
            }
            s_mode = mode;
            s_limit = m_u / a.alpha;
            s_late = late;
        }
    }
    __syncthreads();
    if (s_mode == kTopDown) level_top_down(a, d, s_gr, s_limit, s_mem);
    else if (s_mode == kBottomUp)
        level_bottom_up(a, d, rowptr, cols, front, visited, next, third, parent, level, s_late, s_mem);
}

// The buffers of k_level's levels; false if the memory is not there (the host
// drives the levels then).
bool level_buffers(g5_bfs *b)
{
    if (b->d_ctl) return true;
    // twice n / 8 vertices spread evenly: a level that finds more runs on
    // bottom-up
    b->gcap = std::max<int64_t>(kMinQueue, b->g->n_rows / 4 / kGroups);
    hipError_t e = hipMalloc(&b->d_third, (size_t)std::max<int64_t>(b->wc, 1) * 8);
    for (int k = 0; k < 2; ++k) {
        if (e == hipSuccess) e = hipMalloc(&b->d_gq[k], (size_t)(kGroups * b->gcap) * 4);
        if (e == hipSuccess) e = hipMalloc(&b->d_goff[k], (size_t)(kGroups * b->gcap) * 8);
    }
    if (e == hipSuccess) e = hipMalloc(&b->d_ctl, sizeof(LevelCtl));
    if (e == hipSuccess) return true;
    (void)hipGetLastError();
    auto drop = [](auto *&p) {
        if (p) (void)hipFree(p);
        p = nullptr;
    };
    drop(b->d_third);
    for (int k = 0; k < 2; ++k) {
        drop(b->d_gq[k]);
        drop(b->d_goff[k]);
    }
    return false;
}

// The whole search with k_level; levels are launched in batches.
int run_levels(g5_bfs *b, int64_t root)
{
    g5_graph *g = b->g;
    hipStream_t s = b->s;
    LevelArgs a{};
    a.rowptr = g->d_rowptr;
    a.cols = g->d_cols;
    a.visited = b->d_visited;
    uint64_t *bm[3] = {b->d_out, b->d_next, b->d_third};
    auto at = [&](int d) {
        a.front = bm[d % 3];
        a.next = bm[(d + 1) % 3];
        a.third = bm[(d + 2) % 3];
        a.q = b->d_gq[d & 1];
        a.qn = b->d_gq[(d + 1) & 1];
        a.qoff = b->d_goff[d & 1];
        a.qoffn = b->d_goff[(d + 1) & 1];
    };
    at(0);
    a.parent = b->d_parent;
    a.level = b->d_level;
    a.ctl = b->d_ctl;
    a.host = b->h_cnt + kNCnt;
    a.n = g->n_rows;
    a.wc = b->wc;
    a.nnz = g->nnz;
    a.alpha = b->alpha;
    a.beta = b->beta;
    a.gcap = b->gcap;
    *a.host = 0;
    hipLaunchKernelGGL(k_reset, g5::grid_for(a.n / 4, kLvBlock, 4096), kLvBlock, 0, s, a,
                       (const uint64_t *)b->d_isolated, root - g->row_start);
    const int grid = std::max(256, g5::grid_for(a.wc, kLvBlock / 64, kLvGrid));
    // a Kronecker search runs 6 to 9 levels; a level past the end costs about
    // 2 us, a look from the host about 10
    int d = 0;
    for (int batch = 8;; batch = d < 16 ? 4 : std::min(64, batch * 2)) {
        for (int i = 0; i < batch; ++i, ++d) {
            at(d);
            hipLaunchKernelGGL(k_level, grid, kLvBlock, 0, s, a, d,
                               a.rowptr, a.cols, (const uint64_t *)a.front, a.visited, a.next, a.third, a.parent, a.level);
        }
        G5_HIP(hipGetLastError());
        G5_HIP(hipEventRecord(b->ev1, s));
        G5_HIP(hipStreamSynchronize(s));
        if (*a.host) break;
    }
    const int nlevels = (int)*a.host;
    // as a search level by level leaves it: the frontier empty, all merged
    b->depth = nlevels - 1;
    b->d_out = bm[nlevels % 3];
    b->d_next = bm[(nlevels + 1) % 3];
    b->d_third = bm[(nlevels + 2) % 3];
    b->qlen = 0;
    b->queue_ok = true;
    b->qoff_ok = false;
    b->root = root;
    b->inbits_valid = false;
    return G5_OK;
}

}  // namespace

extern "C" int g5_bfs_create(g5_graph *g, g5_bfs **out)
{
    G5_REQUIRE(g && out, G5_E_ARG, "g5_bfs_create: null argument");
    g5_bfs *b = new g5_bfs();
    b->g = g;
    b->wr = g->n_rows / 64;
    b->wc = g->n_cols / 64;
    auto fail = [&](int rc) {
        g5_bfs_free(b);
        return rc;
    };
    hipError_t e = hipStreamCreate(&b->s);
    const int64_t nmax = std::max(g->n_rows, g->n_cols);
    const size_t scr = g5::scan_scratch_words(nmax + 1) + 64;
    if (e == hipSuccess) e = hipMalloc(&b->d_visited, (size_t)std::max<int64_t>(b->wc, 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_out, (size_t)std::max<int64_t>(b->wc, 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_next, (size_t)std::max<int64_t>(b->wc, 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_parent, (size_t)std::max<int64_t>(g->n_cols, 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&b->d_level, (size_t)std::max<int64_t>(g->n_cols, 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&b->d_queue, (size_t)std::max<int64_t>(nmax, 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&b->d_outq, (size_t)std::max<int64_t>(nmax, 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&b->d_qoff, (size_t)(g->n_rows + 2) * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_scratch, scr * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_cnt, kNCnt * 8);
    if (e == hipSuccess) e = hipMalloc(&b->d_part, 4 * kParts * 8);
    static_assert(kParts >= 2 * g5::kTiles && kParts >= kSumGrid, "a sum per workgroup and tile");
    if (e == hipSuccess) e = hipHostMalloc(&b->h_cnt, (kNCnt + 1) * 8, hipHostMallocDefault);  // k_level's end last
    if (e == hipSuccess) e = hipEventCreate(&b->ev0);
    if (e == hipSuccess) e = hipEventCreate(&b->ev1);
    if (e == hipSuccess) e = hipEventCreate(&b->ek0);
    if (e == hipSuccess) e = hipEventCreate(&b->ek1);
    if (e != hipSuccess) return fail(g5::fail_hip(e, "g5_bfs_create allocation", __FILE__, __LINE__));
    if (g->n_rows == g->n_cols && g->row_start == g->col_start && g->n_rows >= g->nglobal) (void)level_buffers(b);
    *out = b;
    return G5_OK;
}

extern "C" int g5_bfs_free(g5_bfs *b)
{
    if (!b) return G5_OK;
    if (b->s) (void)hipStreamSynchronize(b->s);
    void *dev[] = {b->d_visited, b->d_out,     b->d_next, b->d_parent, b->d_level, b->d_queue,
                   b->d_outq,    b->d_qoff,    b->d_scratch, b->d_cnt, b->d_part, b->d_words, b->d_isolated, b->d_inbits,
                   b->d_third,   b->d_gq[0],   b->d_gq[1], b->d_goff[0], b->d_goff[1], b->d_ctl};
    for (void *p : dev)
        if (p) (void)hipFree(p);
    if (b->h_cnt) (void)hipHostFree(b->h_cnt);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->ek0) (void)hipEventDestroy(b->ek0);
    if (b->ek1) (void)hipEventDestroy(b->ek1);
    b->codec.release();
    if (b->s) (void)hipStreamDestroy(b->s);
    delete b;
    return G5_OK;
}

extern "C" int g5_bfs_start(g5_bfs *b, int64_t root)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_start: null handle");
    int rc = reset_search(b, root);
    if (rc) return rc;
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_expand(g5_bfs *b, int *any_new)
{
    G5_REQUIRE(b && any_new, G5_E_ARG, "g5_bfs_expand: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_expand: g5_bfs_start not called");
    int rc = prepare_queue(b, b->d_out);
    if (!rc) rc = expand_level(b, b->d_out, true, -1);
    // the out bits are this block's newly reached columns
    const int slot[] = {kOutLen};
    if (!rc && b->prof) G5_HIP(hipMemcpyAsync(b->h_cnt, b->d_cnt, 2 * 8, hipMemcpyDeviceToHost, b->s));
    if (!rc) rc = fold_counters(b, kParts, kExpandGrid, slot, 1, false);
    if (!rc) rc = account_level(b, b->h_cnt[kQLen], b->h_cnt[kEdges], b->h_cnt[kOutLen]);
    if (rc) return rc;
    *any_new = b->h_cnt[kOutLen] > 0;
    return G5_OK;
}

extern "C" int g5_bfs_outqueue(g5_bfs *b, uint32_t *q, int64_t *n)
{
    G5_REQUIRE(b && n, G5_E_ARG, "g5_bfs_outqueue: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_outqueue: g5_bfs_start not called");
    g5::QueueOut o{};
    o.q = b->d_outq;
    o.h_n = b->h_cnt + kOutLen;
    G5_HIP(g5::bitmap_to_queue(b->d_out, b->wc, nullptr, o, b->d_part, false, b->s));
    G5_HIP(hipStreamSynchronize(b->s));
    const int64_t len = b->h_cnt[kOutLen];
    G5_REQUIRE(len <= *n, G5_E_OVERFLOW, "g5_bfs_outqueue: queue of %lld entries exceeds capacity %lld",
               (long long)len, (long long)*n);
    *n = len;
    if (len) {
        G5_REQUIRE(q, G5_E_ARG, "g5_bfs_outqueue: null queue buffer");
        G5_HIP(hipMemcpy(q, b->d_outq, (size_t)len * 4, hipMemcpyDeviceToHost));
    }
    return G5_OK;
}

// the level's newly reached columns: bits, which may be d_out
static hipError_t commit_out(g5_bfs *b, const uint64_t *bits)
{
    if (b->wc == 0) return hipSuccess;
    hipLaunchKernelGGL(k_commit, g5::tile_count(b->wc), 256, 0, b->s, bits, b->d_out, b->d_visited, b->d_level, b->wc,
                       g5::tile_words(b->wc), (int32_t)(b->depth + 1), (const int64_t *)nullptr, (int64_t *)nullptr);
    return hipGetLastError();
}

extern "C" int g5_bfs_set_outqueue(g5_bfs *b, const uint32_t *q, int64_t n)
{
    G5_REQUIRE(b && n >= 0, G5_E_ARG, "g5_bfs_set_outqueue: bad arguments");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_set_outqueue: g5_bfs_start not called");
    g5_graph *g = b->g;
    if (q) {
        G5_REQUIRE(n <= g->n_cols, G5_E_OVERFLOW, "g5_bfs_set_outqueue: queue longer than the column slice");
        for (int64_t i = 0; i < n; ++i)
            G5_REQUIRE(q[i] < (uint64_t)g->n_cols && (i == 0 || q[i] > q[i - 1]), G5_E_ARG,
                       "g5_bfs_set_outqueue: queue not sorted/unique/in range at %lld", (long long)i);
        G5_HIP(g5::fill_u64(b->d_out, b->wc, 0, b->s));
        if (n) {
            G5_HIP(hipMemcpyAsync(b->d_outq, q, (size_t)n * 4, hipMemcpyHostToDevice, b->s));
            G5_HIP(g5::queue_to_bitmap(b->d_outq, n, b->d_out, b->wc, nullptr, b->s));
        }
    }
    G5_HIP(commit_out(b, b->d_out));
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_set_inqueue(g5_bfs *b, const uint32_t *q, int64_t n)
{
    G5_REQUIRE(b && n >= 0, G5_E_ARG, "g5_bfs_set_inqueue: bad arguments");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_set_inqueue: g5_bfs_start not called");
    g5_graph *g = b->g;
    if (q) {
        G5_REQUIRE(n <= g->n_rows, G5_E_OVERFLOW, "g5_bfs_set_inqueue: queue longer than the row slice");
        for (int64_t i = 0; i < n; ++i)
            G5_REQUIRE(q[i] < (uint64_t)g->n_rows && (i == 0 || q[i] > q[i - 1]), G5_E_ARG,
                       "g5_bfs_set_inqueue: queue not sorted/unique/in range at %lld", (long long)i);
        if (n) G5_HIP(hipMemcpyAsync(b->d_queue, q, (size_t)n * 4, hipMemcpyHostToDevice, b->s));
        b->qlen = n;
        b->qoff_ok = false;
    } else {
        G5_REQUIRE(g->n_rows == g->n_cols && g->row_start == g->col_start, G5_E_STATE,
                   "g5_bfs_set_inqueue: own out-queue as in-queue needs a diagonal block");
        g5::QueueOut o{};
        o.q = b->d_queue;
        o.qoff = b->d_qoff;
        o.d_n = b->d_cnt + kQLen;
        o.d_e = b->d_cnt + kEdges;
        o.h_n = b->h_cnt + kQLen;
        G5_HIP(g5::bitmap_to_queue(b->d_out, b->wc, (const int64_t *)g->d_rowptr, o, b->d_part, false, b->s));
        b->qoff_ok = true;
    }
    G5_HIP(hipStreamSynchronize(b->s));
    if (!q) b->qlen = b->h_cnt[kQLen];
    b->queue_ok = true;
    b->inbits_valid = false;
    b->depth++;
    return G5_OK;
}

extern "C" int g5_bfs_result(g5_bfs *b, int64_t *pred, int32_t *level)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_result: null handle");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_result: no search");
    g5_graph *g = b->g;
    if (pred) {
        int64_t *d = nullptr;
        G5_HIP(hipMallocAsync((void **)&d, (size_t)std::max<int64_t>(g->n_cols, 1) * 8, b->s));
        hipLaunchKernelGGL(k_result, g5::grid_for(g->n_cols, 256, 8192), 256, 0, b->s,
                           (const uint32_t *)b->d_parent, g->n_cols, g->row_start, g->col_start, d);
        G5_HIP(hipGetLastError());
        G5_HIP(hipMemcpyAsync(pred, d, (size_t)g->n_cols * 8, hipMemcpyDeviceToHost, b->s));
        G5_HIP(hipFreeAsync(d, b->s));
    }
    if (level) G5_HIP(hipMemcpyAsync(level, b->d_level, (size_t)g->n_cols * 4, hipMemcpyDeviceToHost, b->s));
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_out_bitmap(g5_bfs *b, const uint64_t **d_bits, int64_t *n_words)
{
    G5_REQUIRE(b && d_bits && n_words, G5_E_ARG, "g5_bfs_out_bitmap: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_out_bitmap: g5_bfs_start not called");
    *d_bits = b->d_out;
    *n_words = b->wc;
    return G5_OK;
}

extern "C" int g5_bfs_set_out_bitmap(g5_bfs *b, const uint64_t *d_bits)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_set_out_bitmap: null handle");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_set_out_bitmap: g5_bfs_start not called");
    // bits in this GPU's memory are read where they lie
    if (d_bits && b->wc && d_bits != b->d_out && !g5::in_memory_of(b->g->device, d_bits, b->wc)) {
        G5_HIP(hipMemcpyAsync(b->d_out, d_bits, (size_t)b->wc * 8, hipMemcpyDefault, b->s));
        d_bits = b->d_out;
    }
    G5_HIP(commit_out(b, d_bits && b->wc ? d_bits : b->d_out));
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_set_in_bitmap(g5_bfs *b, const uint64_t *d_bits)
{
    G5_REQUIRE(b && d_bits, G5_E_ARG, "g5_bfs_set_in_bitmap: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_set_in_bitmap: g5_bfs_start not called");
    if (!b->d_inbits) G5_HIP(hipMalloc(&b->d_inbits, (size_t)(b->wr ? b->wr : 1) * 8));
    // the queue is made by an expansion that runs top-down, which needs it
    if (g5::in_memory_of(b->g->device, d_bits, b->wr)) {
        hipLaunchKernelGGL(k_copy_words, g5::grid_for(b->wr, 256, 4096), 256, 0, b->s, d_bits, b->d_inbits, b->wr);
        G5_HIP(hipGetLastError());
    } else if (b->wr) {
        G5_HIP(hipMemcpyAsync(b->d_inbits, d_bits, (size_t)b->wr * 8, hipMemcpyDefault, b->s));
    }
    G5_HIP(hipStreamSynchronize(b->s));
    b->queue_ok = b->qoff_ok = false;
    b->inbits_valid = true;
    b->depth++;
    return G5_OK;
}

extern "C" int g5_bfs_expand_bottom_up(g5_bfs *b, const g5_graph *gt, int *any_new)
{
    G5_REQUIRE(b && gt && any_new, G5_E_ARG, "g5_bfs_expand_bottom_up: null argument");
    G5_REQUIRE(b->depth >= 0 && b->inbits_valid, G5_E_STATE,
               "g5_bfs_expand_bottom_up: needs a row frontier from g5_bfs_set_in_bitmap");
    const g5_graph *g = b->g;
    G5_REQUIRE(gt->n_rows == g->n_cols && gt->n_cols == g->n_rows && gt->row_start == g->col_start &&
                   gt->col_start == g->row_start,
               G5_E_ARG, "g5_bfs_expand_bottom_up: gt is not the transposed block");
    hipStream_t s = b->s;
    if (b->prof) G5_HIP(hipEventRecord(b->ek0, s));
    // rows of gt = this block's columns, its columns = this block's rows: the
    // kernel's frontier bits are the row frontier, its parents local row ids
    const int grid = g5::grid_for(b->wc, 4, kParts);
    hipLaunchKernelGGL(k_bottom_up<false>, grid, 256, 0, s, (const int64_t *)gt->d_rowptr,
                       (const uint32_t *)gt->d_cols, b->d_visited, (const uint64_t *)b->d_inbits, b->d_out,
                       b->d_parent, (int32_t *)nullptr, 0, b->wc, b->d_part);
    G5_HIP(hipGetLastError());
    if (b->prof) G5_HIP(hipEventRecord(b->ek1, s));
    const int slot[] = {kOutLen, kNewEdges, kBuEdges, kBuVerts};
    int rc = fold_counters(b, kParts, grid, slot, 4, false);
    if (!rc) rc = account_bottom_up(b, b->h_cnt[kOutLen], false);
    if (rc) return rc;
    *any_new = b->h_cnt[kOutLen] > 0;
    return G5_OK;
}

extern "C" int g5_bfs_pred_device(g5_bfs *b, int64_t *d_pred)
{
    G5_REQUIRE(b && d_pred, G5_E_ARG, "g5_bfs_pred_device: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_pred_device: no search");
    g5_graph *g = b->g;
    hipLaunchKernelGGL(k_result, g5::grid_for(g->n_cols, 256, 8192), 256, 0, b->s, (const uint32_t *)b->d_parent,
                       g->n_cols, g->row_start, g->col_start, d_pred);
    G5_HIP(hipGetLastError());
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_level_device(g5_bfs *b, int32_t *d_level)
{
    G5_REQUIRE(b && d_level, G5_E_ARG, "g5_bfs_level_device: null argument");
    G5_REQUIRE(b->depth >= 0, G5_E_STATE, "g5_bfs_level_device: no search");
    G5_HIP(hipMemcpyAsync(d_level, b->d_level, (size_t)b->g->n_cols * 4, hipMemcpyDeviceToDevice, b->s));
    G5_HIP(hipStreamSynchronize(b->s));
    return G5_OK;
}

extern "C" int g5_bfs_nedge(g5_bfs *b, int64_t *nedge)
{
    G5_REQUIRE(b && nedge, G5_E_ARG, "g5_bfs_nedge: null argument");
    G5_REQUIRE(b->g->n_rows == b->g->n_cols, G5_E_STATE, "g5_bfs_nedge: needs a 1x1 block");
    const int grid = g5::grid_for(b->g->n_rows / 4, 256, kSumGrid);
    hipLaunchKernelGGL(k_nedge, grid, 256, 0, b->s, (const uint32_t *)b->g->d_gdeg, (const int32_t *)b->d_level,
                       b->g->n_rows, b->d_part);
    G5_HIP(hipGetLastError());
    const int slot[] = {kOutLen};
    int rc = fold_counters(b, kParts, grid, slot, 1, false);
    if (rc) return rc;
    *nedge = b->h_cnt[kOutLen] / 2;
    return G5_OK;
}

extern "C" int g5_bfs_summary(g5_bfs *b, int64_t *nedge, uint64_t *checksum)
{
    G5_REQUIRE(b && nedge && checksum, G5_E_ARG, "g5_bfs_summary: null argument");
    G5_REQUIRE(b->g->n_rows == b->g->n_cols && b->g->row_start == b->g->col_start, G5_E_STATE,
               "g5_bfs_summary: needs a diagonal (1x1) block");
    const int grid = g5::grid_for(b->g->n_rows, 256, kSumGrid);
    hipLaunchKernelGGL(k_summary, grid, 256, 0, b->s, (const uint32_t *)b->g->d_gdeg, (const int32_t *)b->d_level,
                       (const uint32_t *)b->d_parent, b->g->n_rows, b->d_part);
    G5_HIP(hipGetLastError());
    const int slot[] = {kOutLen, kNewEdges};
    int rc = fold_counters(b, kParts, grid, slot, 2, false);
    if (rc) return rc;
    *nedge = b->h_cnt[kOutLen] / 2;
    *checksum = (uint64_t)b->h_cnt[kNewEdges];
    return G5_OK;
}

extern "C" int g5_bfs_run(g5_bfs *b, int64_t root, int flags, int32_t *nlevels, float *ms)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_run: null handle");
    g5_graph *g = b->g;
    G5_REQUIRE(g->n_rows == g->n_cols && g->row_start == g->col_start, G5_E_STATE,
               "g5_bfs_run: the resident loop needs a diagonal (1x1) block");
    G5_REQUIRE(root >= 0 && root < g->n_rows, G5_E_ARG, "g5_bfs_run: root %lld out of range", (long long)root);
    const bool codec = (flags & G5_RUN_CODEC) != 0;
    const bool topdown_only = (flags & G5_RUN_TOPDOWN) != 0;
    if (codec && !b->d_words) {
        b->words_cap = g5_s4_max_words((size_t)g->n_cols);
        G5_HIP(hipMalloc(&b->d_words, b->words_cap * 4));
        int rc = b->codec.reserve((int64_t)g->n_cols);
        if (rc) return rc;
    }
    // k_level decides the levels on the device; the codec's launches, the
    // accounting and a forced direction need the host's view of each level,
    // a packed total holds 2^30 vertices and 2^34 edges, and a root outside the
    // block (one that does not start at vertex 0) has no row to start from
    const bool here = root >= g->row_start && root - g->row_start < g->n_rows;
    const bool on_device = !codec && !topdown_only && !b->prof && here && g->n_rows <= (int64_t)1 << 30 &&
                           g->nnz < (int64_t)1 << kEdgeBits && level_buffers(b);
    hipStream_t s = b->s;
    G5_HIP(hipStreamSynchronize(s));
    G5_HIP(hipEventRecord(b->ev0, s));  // a first search's time holds the look for edgeless vertices
    int rc = find_isolated(b);
    if (rc) return rc;
    if (on_device) {
        rc = run_levels(b, root);
        if (rc) return rc;
        if (ms) G5_HIP(hipEventElapsedTime(ms, b->ev0, b->ev1));
        if (nlevels) *nlevels = b->depth + 1;
        return G5_OK;
    }
    rc = reset_search(b, root, true);
    if (rc) return rc;
    const int64_t n = g->n_rows;
    int64_t m_u = g->nnz;  // edges not yet checked top-down
    bool bu = false;       // the first level is always top-down
    int64_t E = 0;         // the frontier's edges
    if (b->prof) G5_HIP(hipMemcpyAsync(&b->h_cnt[kEdges], b->d_cnt + kEdges, 8, hipMemcpyDeviceToHost, s));
    const int64_t tile = g5::tile_words(b->wc);
    const int tiles = g5::tile_count(b->wc), bu_grid = g5::grid_for(b->wc, 4, kParts);
    // d_out is the frontier, d_next the next one (clear before a top-down level)
    for (;;) {
        if (bu) {
            if (b->prof) G5_HIP(hipEventRecord(b->ek0, s));
            hipLaunchKernelGGL(k_bottom_up<true>, bu_grid, 256, 0, s, (const int64_t *)g->d_rowptr,
                               (const uint32_t *)g->d_cols, b->d_visited, (const uint64_t *)b->d_out, b->d_next,
                               b->d_parent, b->d_level, (int32_t)(b->depth + 1), b->wc, b->d_part);
            G5_HIP(hipGetLastError());
            if (b->prof) G5_HIP(hipEventRecord(b->ek1, s));
            const int slot[] = {kNew, kNewEdges, kBuEdges, kBuVerts};
            rc = fold_counters(b, kParts, bu_grid, slot, 4, true);
        } else {
            rc = expand_level(b, b->d_next, false, b->depth == 0 ? -1 : E);
            if (rc) return rc;
            hipLaunchKernelGGL(k_commit, tiles, 256, 0, s, (const uint64_t *)b->d_next, b->d_next, b->d_visited,
                               b->d_level, b->wc, tile, (int32_t)(b->depth + 1), (const int64_t *)g->d_rowptr,
                               b->d_part);
            G5_HIP(hipGetLastError());
            const int slot[] = {kNew, kNewEdges};
            rc = fold_counters(b, g5::kTiles, tiles, slot, 2, true);
        }
        if (rc) return rc;
        std::swap(b->d_out, b->d_next);
        // the previous level's codec round trip has completed by now
        G5_REQUIRE(b->h_cnt[kCodecErr] == 0, G5_E_STREAM, "g5_bfs_run: codec round trip lost values");
        const int64_t n_new = b->h_cnt[kNew];
        if (b->depth == 0) E = b->h_cnt[kEdges];
        rc = bu ? account_bottom_up(b, n_new, true) : account_level(b, b->qlen, E, n_new);
        if (rc) return rc;
        if (n_new == 0) break;
        // the next level's direction
        const int64_t m_f = b->h_cnt[kNewEdges];
        bool bu_next = bu;
        if (!topdown_only) {
            if (!bu && m_f > m_u / b->alpha) bu_next = true;
            else if (bu && n_new < n / b->beta) bu_next = false;
        }
        if (!bu_next) m_u -= m_f;
        // the out-bitmap holds exactly the new vertices; a queue of them is
        // needed by a top-down level and by the codec
        b->qlen = n_new;
        E = m_f;
        if (!bu_next || codec) {
            g5::QueueOut o{};
            o.q = b->d_queue;
            o.qoff = b->d_qoff;
            o.clear = b->d_next;
            o.n_clear = bu_next ? 0 : b->wc;
            // a top-down level's commit has left its tiles' sums
            G5_HIP(g5::bitmap_to_queue(b->d_out, b->wc, bu_next ? nullptr : (const int64_t *)g->d_rowptr, o,
                                       b->d_part, !bu, s));
        }
        if (codec) {
            // encode -> decode in place with no host synchronisation; checked
            // at the next level's counter read
            rc = b->codec.roundtrip(b->d_queue, b->qlen, b->d_words, b->words_cap, b->d_queue, b->d_cnt + kCodecErr, s);
            if (rc) return rc;
        }
        bu = bu_next;
        b->depth++;
    }
    G5_HIP(hipEventRecord(b->ev1, s));
    G5_HIP(hipEventSynchronize(b->ev1));
    if (ms) G5_HIP(hipEventElapsedTime(ms, b->ev0, b->ev1));
    if (nlevels) *nlevels = b->depth + 1;
    // no frontier is left
    b->qlen = 0;
    b->queue_ok = true;
    b->qoff_ok = false;
    return G5_OK;
}

extern "C" int g5_bfs_tune(g5_bfs *b, int64_t alpha, int64_t beta)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_tune: null handle");
    G5_REQUIRE(alpha >= 1 && beta >= 1, G5_E_ARG, "g5_bfs_tune: alpha and beta must be >= 1");
    b->alpha = alpha;
    b->beta = beta;
    return G5_OK;
}

extern "C" int g5_bfs_profile(g5_bfs *b, int enable)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_profile: null handle");
    b->prof = enable != 0;
    b->exp_ms = b->exp_bytes = 0;
    b->exp_launches = b->exp_edges = 0;
    b->bu_ms = b->bu_bytes = 0;
    b->bu_launches = b->bu_edges = 0;
    return G5_OK;
}

extern "C" int g5_bfs_kernel_stats(g5_bfs *b, int kernel, double *ms, int64_t *launches, double *bytes,
                                   int64_t *edges)
{
    G5_REQUIRE(b && (kernel == 0 || kernel == 1), G5_E_ARG, "g5_bfs_kernel_stats: kernel must be 0 or 1");
    if (kernel == 0) return g5_bfs_stats(b, ms, launches, bytes, edges);
    if (ms) *ms = b->bu_ms;
    if (launches) *launches = b->bu_launches;
    if (bytes) *bytes = b->bu_bytes;
    if (edges) *edges = b->bu_edges;
    return G5_OK;
}

extern "C" int g5_bfs_stats(g5_bfs *b, double *ms, int64_t *launches, double *bytes, int64_t *edges)
{
    G5_REQUIRE(b, G5_E_ARG, "g5_bfs_stats: null handle");
    if (ms) *ms = b->exp_ms;
    if (launches) *launches = b->exp_launches;
    if (bytes) *bytes = b->exp_bytes;
    if (edges) *edges = b->exp_edges;
    return G5_OK;
}
