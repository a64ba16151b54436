// bfs_device.hpp -- gfx950 device building blocks of the BFS kernels.
//
// Wave64 primitives (DPP prefix sum, ballot/mbcnt compaction), the per-wave
// LDS-staged frontier queue, the visited-bitmask claims, the workgroup
// neighbour gather and the hierarchical grid barrier.  These replace the
// reference's CTA raking scans, warp scans, tile I/O, culls and software
// global barrier (b40c/util/scan/*.cuh, b40c/util/io/*.cuh,
// b40c/util/global_barrier.cuh, b40c/graph/bfs/*/cta.cuh); the designs are
// written for 64-lane waves and CDNA memory scopes, not translated.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace b40c_hip {

constexpr int kWave = 64;
constexpr int kHistory = 1024;                 // LDS history-hash entries per workgroup
constexpr int kBarrierFanIn = 16;              // first-level barrier counters
constexpr int kHubChunk = 2048;                // edges per grid-tier chunk
constexpr int kLevelLog = 64;                  // steps with recorded length/clock

// ---------------------------------------------------------------------------
// Device control block: frontier lengths, tile counters, barrier state, exit
// status.  Counters rotate by step so a step never zeroes a counter that is
// still being read: step s reads qlen[s % 3], appends to qlen[(s+1) % 3] and
// zeroes qlen[(s+2) % 3] and steal[(s+1) & 1].
// ---------------------------------------------------------------------------
struct alignas(256) Control {
    unsigned qlen[4];
    unsigned steal[2];
    unsigned overflow;
    int exit_reason;          // 0 done, 1 saturated, 2 overflow
    int exit_step;            // loop position when a persistent launch ends
    int exit_iteration;
    int exit_phase;
    int fast_step;            // single-workgroup fast path hand-off
    int fast_iteration;
    int fast_phase;
    int max_depth;            // deepest label written
    unsigned compact;         // bitmap -> queue reservations (zeroed every step)
    unsigned long long total_queued;
    unsigned long long busy_cycles;   // instrumented: sum over workgroups of step time
    unsigned long long life_cycles;   // instrumented: sum over workgroups of kernel time
    unsigned long long hub_alloc[2];  // grid tier: (entries << 32) | chunks, by step & 1
    unsigned hub_steal[2];            // grid tier: chunk counter, by step & 1
    unsigned hybrid_stop;             // hybrid two-phase launches: the filtered frontier fits the
                                      // persistent kernel again (exit_step / exit_iteration say where)
    unsigned pad1[3];
    // Direction-optimizing bookkeeping (second 128-byte line).
    unsigned long long fedges[3];     // sum of degrees of each frontier, by step % 3
    unsigned long long visited_edges; // launches per step: sum of fedges over the steps before the current one
    unsigned long long fast_vsum;     // fast-path hand-off of the per-workgroup visited-edge sum
    unsigned ovf[4];                  // per-step overflow of the output queue, by step % 3
    unsigned long long fast_prev_fe;  // fast-path hand-off: frontier edges of the level before the next step's
    unsigned long long pad2[8];
    unsigned bar_root;        // own 128-byte line
    unsigned pad3[31];
    unsigned bar_gen;         // completed barriers (own 128-byte line)
    unsigned pad4[31];
    unsigned bar_leaf[kBarrierFanIn * 32];     // one 128-byte line per leaf counter
    unsigned bar_release[kBarrierFanIn * 32];  // one 128-byte line per leaf release word
    unsigned level_len[kLevelLog];             // input length of each step
    unsigned long long level_clock[kLevelLog]; // wall clock at the start of each step
};

// Bytes of the control block's status head (counters, flags, statistics):
// what the host reads after a search or a step.
constexpr size_t kControlHead = 256;
static_assert(offsetof(Control, bar_root) == kControlHead, "status head ends where the barrier lines begin");

// Grid-tier work item: a row too long for one workgroup, split into
// kHubChunk-edge chunks [first_chunk, first_chunk + ceil(len / kHubChunk)).
struct HubEntry {
    int beg, end, par;
    unsigned first_chunk;
    int tag;   // batched searches: the query; expansions: the row's place in the output queue
};

enum ExitReason { kExitDone = 0, kExitSaturated = 1, kExitOverflow = 2 };

// ---------------------------------------------------------------------------
// Threads per workgroup, chosen per translation unit.  The single-source
// kernels run 512: a grid barrier's release and acquire fences cost about
// the same per workgroup, so fewer, larger workgroups halve its cost at the
// same wave count.  The batch kernels build with 256 (B40C_BLOCK=256).
// Everything below depends on it and sits in an inline namespace named
// after the size, so the two builds never share a symbol.
// ---------------------------------------------------------------------------
#ifndef B40C_BLOCK
#define B40C_BLOCK 512
#endif
#define B40C_NS_CAT2(a, b) a##b
#define B40C_NS_CAT(a, b) B40C_NS_CAT2(a, b)
inline namespace B40C_NS_CAT(block, B40C_BLOCK) {

constexpr int kBlock = B40C_BLOCK;
constexpr int kWaves = kBlock / kWave;         // waves per workgroup
static_assert(kBlock % kWave == 0 && kBlock >= 128 && kBlock <= 1024, "workgroup of whole waves");

// LDS staging entries per wave of the frontier queues.  Every full area
// costs one reservation atomic on the queue's length, and on a large
// level those atomics, all on one address, bound the step: 2048 entries
// per wave took the single-source two-phase search on R-MAT s22 from 5.09
// to 2.64 ms (64 KiB of LDS per 512-thread workgroup, 128 KiB with the
// predecessor staging).  The batch kernels keep 512, which leaves them
// their occupancy of three 256-thread workgroups per CU.
constexpr int kWaveQueueCap = kBlock >= 512 ? 2048 : 512;

// ---------------------------------------------------------------------------
// Wave64 primitives
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane_id()
{
    return (int) __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// Number of set bits of `m` below the calling lane.
__device__ __forceinline__ int lanes_below(uint64_t m)
{
    return (int) __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32),
                                           __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ int readlane(int x, int l) { return __builtin_amdgcn_readlane(x, l); }

// Inclusive prefix sum across the 64 lanes with DPP row shifts inside each
// 16-lane row followed by the row_bcast:15 / row_bcast:31 carries between
// rows (GFX9/CDNA DPP controls 0x111..0x118, 0x142, 0x143).  Lanes whose
// DPP source is out of the row, or whose row is masked off, add 0.
__device__ __forceinline__ int wave_inclusive_sum(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 -> rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 -> rows 2, 3
    return x;
}

// Inclusive running maximum of non-negative values across the 64 lanes (the
// same DPP steps; lanes with no source take 0, the identity here).  The last
// lane holds the wave's maximum.
__device__ __forceinline__ int wave_inclusive_max_nonneg(int x)
{
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false));
    return x;
}

// Exclusive prefix sum over the workgroup (one value per thread): wave DPP
// sums, then the four wave totals through LDS.
__device__ __forceinline__ int block_exclusive_sum(int x, int *wave_tot, int *total)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int incl = wave_inclusive_sum(x);
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    int off = 0, tot = 0;
    for (int w = 0; w < kWaves; w++) {
        int t = wave_tot[w];
        if (w < wave) off += t;
        tot += t;
    }
    *total = tot;
    __syncthreads();
    return off + incl - x;
}

// ---------------------------------------------------------------------------
// Scoped memory helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned ld_agent(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int ld_agent(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Queue entries another workgroup stored in an earlier step, read once:
// system scope makes the load miss in every cache level, so a line this XCD
// still holds from an older use of the buffer (an earlier step or search)
// cannot be returned.  Streamed data, so nothing is lost by not caching it.
__device__ __forceinline__ int ld_queue(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void st_agent(unsigned *p, unsigned v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned add_agent(unsigned *p, unsigned v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Visited claims.
//
// Exact: the bitmask word is first read with a plain (cacheable, possibly
// stale) load.  Bits only ever go 0 -> 1 during a search, so a set bit is
// always true and skips the atomic; a clear bit may be stale and is settled
// by the agent-scope atomic OR, whose returned old value makes exactly one
// claimant the owner of the vertex.
//
// Best effort (the reference discipline, contract_expand_atomic/cta.cuh:
// 213-304): racy read-modify-write of the mask byte as a pre-filter, then the
// label check; racing discoverers may both succeed, which only duplicates
// work because they write the same depth.
// ---------------------------------------------------------------------------
// The pre-test read decides only whether to try the atomic.  The cached read
// may miss bits other workgroups set during this level (device-scope atomics
// are performed beyond this XCD's L2, which keeps its old copy); the
// coherent read sees them at the cost of a longer trip.
__device__ __forceinline__ bool claim_exact(unsigned *visited, int u, bool coherent = false)
{
    unsigned *w = visited + (u >> 5);
    unsigned bit = 1u << (u & 31);
    unsigned cur = coherent ? __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *w;
    if (cur & bit) return false;
    unsigned old = __hip_atomic_fetch_or(w, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (old & bit) == 0;
}

__device__ __forceinline__ bool claim_best_effort(unsigned *visited, const int *depth, int u)
{
    unsigned *w = visited + (u >> 5);
    unsigned bit = 1u << (u & 31);
    unsigned cur = *w;
    if (cur & bit) return false;
    *w = cur | bit;
    return depth[u] == -1;
}

template <bool EXACT>
__device__ __forceinline__ bool claim(unsigned *visited, const int *depth, int u, bool coherent = false)
{
    if (EXACT) return claim_exact(visited, u, coherent);
    return claim_best_effort(visited, depth, u);
}

// ---------------------------------------------------------------------------
// LDS layout shared by every BFS kernel.
// ---------------------------------------------------------------------------
template <bool PRED>
struct PredStore {
    int buf[kWaves][kWaveQueueCap];
};
template <>
struct PredStore<false> {
    int buf[1][1];
};

// Row table of gather_tile, in parts a wave can use by itself.
struct RowTable {
    int excl[kWaves][kWave];             // edge offset
    int beg[kWaves][kWave];              // row begin (gather_tile: less the edge offset)
    int par[kWaves][kWave];              // row owner
    int scan[kWaves], scan2[kWaves];
    int end;                             // end of the table's edges
};

template <bool PRED>
struct Lds {
    int wq[kWaves][kWaveQueueCap];       // per-wave frontier staging
    PredStore<PRED> wqp;                 // per-wave predecessor staging
    RowTable rt;
    int hist[kHistory];                  // history hash (contract / filter)
    int cta_beg, cta_end, cta_par;
    unsigned cta_out;                    // expansions: the chunk's place in the output queue
    unsigned tile;
    unsigned nb;                         // broadcast frontier length
    int step, iteration;
    // end-of-step reduction over the waves (one global update per workgroup)
    unsigned ep_count[kWaves];
    unsigned ep_extra[kWaves];
    unsigned long long ep_fe[kWaves];
    int ep_lab[kWaves];
    int ep_scan[kWaves];
    unsigned ep_base;
    int solo;                            // 1: this workgroup runs the step alone (no static tiles)
};

// ---------------------------------------------------------------------------
// Per-wave frontier queue.  Lanes append through ballot + mbcnt into the
// wave's LDS staging area; a full area (or the end of a step) is flushed with
// one agent-scope atomic reservation and coalesced stores.  One global atomic
// per kWaveQueueCap appended elements (or per wave per step) replaces the
// reference's per-tile raking scan + atomicAdd (util/scan/cooperative_scan.cuh:
// 172-195, 309-343).
// ---------------------------------------------------------------------------
template <bool PRED>
struct WaveQueue {
    int *buf;
    int *pbuf;
    int count;          // wave-uniform
    int *out;
    int *pout;
    unsigned *out_len;
    unsigned cap;
    unsigned *overflow;
    unsigned *overflow_step;   // per-step flag the level loop decides on (may alias overflow)
    bool through;              // a light barrier follows: entries go past the L2 (agent-scope stores)

    __device__ __forceinline__ void store(unsigned at, int u, int p)
    {
        if (through) {
            st_agent(out + at, u);
            if (PRED) st_agent(pout + at, p);
        } else {
            out[at] = u;
            if (PRED) pout[at] = p;
        }
    }

    __device__ __forceinline__ void flush()
    {
        if (count == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        int lane = lane_id();
        unsigned base = 0;
        if (lane == 0) base = add_agent(out_len, (unsigned) count);
        base = (unsigned) uniform((int) base);
        unsigned lim = 0;
        if (base < cap) lim = min((unsigned) count, cap - base);
        if (lim < (unsigned) count && lane == 0) {
            st_agent(overflow, 1u);
            st_agent(overflow_step, 1u);
        }
        for (unsigned i = lane; i < lim; i += kWave) store(base + i, buf[i], PRED ? pbuf[i] : -1);
        count = 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // Wave-converged: every lane of the wave calls push together.
    __device__ __forceinline__ void push(bool flag, int u, int p)
    {
        uint64_t m = ballot(flag);
        if (m == 0) return;
        int c = __popcll(m);
        if (count + c > kWaveQueueCap) flush();
        if (flag) {
            int pos = count + lanes_below(m);
            buf[pos] = u;
            if (PRED) pbuf[pos] = p;
        }
        count += c;
    }
};

// Grid tier of a gathering step: where its long rows are published.
struct HubList {
    HubEntry *entries;
    unsigned cap;
    unsigned long long *alloc;
    int grid_t;        // rows at least this long go to the grid tier
    int tag;           // stored with every published row
    unsigned *out_len; // expansions: length of the output queue (null: none reserved)
    int heavy, heavy_row;  // edges from which a tile publishes its rows of heavy_row and more (gather_tile)
};

// Index of the last grid-tier entry whose first chunk is <= ch (entries are
// in chunk order).  A workgroup takes chunks in increasing order, so the
// search gallops forward from the entry of its previous chunk (`hint`): the
// next chunk usually lies in the same entry or the next one, one or two
// loads instead of a binary search's chain of dependent loads.
__device__ __forceinline__ unsigned hub_entry_of(const HubEntry *list, unsigned entries, unsigned ch, unsigned hint)
{
    unsigned lo = 0, hi = entries - 1;
    if (hint < entries && list[hint].first_chunk <= ch) {
        lo = hint;
        unsigned step = 1;
        while (lo + step < entries && list[lo + step].first_chunk <= ch) {
            lo += step;
            step <<= 1;
        }
        hi = min(lo + step, entries) - 1;
    }
    while (lo < hi) {
        const unsigned mid = (lo + hi + 1) >> 1;
        if (list[mid].first_chunk <= ch) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Grid-tier publication of a row of at least hub.grid_t neighbours (called
// wave-converged; true when this lane's row was published).  The wave
// reserves list entries and chunk numbers for all its long rows with one
// atomic; entries keep lane order, so the list stays sorted by first chunk.
// With hub.out_len set, the wave also reserves that many elements of the
// output queue for its published rows (one more atomic), and an entry's tag
// is its row's place there: the grid tier then writes without reserving.
__device__ __forceinline__ bool publish_hub_row(int beg, int end, int par, const HubList &hub)
{
    const int lane = lane_id();
    const int len = end - beg;
    const bool pub = len >= hub.grid_t;
    const uint64_t pm = ballot(pub);
    if (!pm) return false;
    const int nch = pub ? (len + kHubChunk - 1) / kHubChunk : 0;
    const int incl = wave_inclusive_sum(nch);
    const unsigned total = (unsigned) readlane(incl, kWave - 1);
    unsigned lo = 0, hi = 0;
    if (lane == 0) {
        unsigned long long old = __hip_atomic_fetch_add(hub.alloc, ((unsigned long long) __popcll(pm) << 32) | total,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lo = (unsigned) old;
        hi = (unsigned) (old >> 32);
    }
    lo = (unsigned) uniform((int) lo);
    hi = (unsigned) uniform((int) hi);
    const unsigned slot = hi + (unsigned) lanes_below(pm);
    const bool done = pub && slot < hub.cap;
    int tag = hub.tag;
    if (hub.out_len) {
        const int lens = wave_inclusive_sum(done ? len : 0);
        unsigned at = 0;
        if (lane == kWave - 1) at = add_agent(hub.out_len, (unsigned) lens);
        tag = (int) ((unsigned) readlane((int) at, kWave - 1) + (unsigned) (lens - len));
    }
    if (done) {
        // (past the L2: a light barrier may follow)
        HubEntry *h = hub.entries + slot;
        st_agent(&h->beg, beg);
        st_agent(&h->end, end);
        st_agent(&h->par, par);
        st_agent(&h->first_chunk, lo + (unsigned) (incl - nch));
        st_agent(&h->tag, tag);
    }
    return done;
}

// ---------------------------------------------------------------------------
// Workgroup gather of a tile of rows.  Each thread brings up to K rows
// [beg, end) with owner par (end == beg for none).  Long rows go to the grid
// tier; the others are compacted into an LDS table of kBlock rows (row start,
// edge offset, owner) and their edges spread evenly over the workgroup: each
// round covers kBlock * 4 consecutive edges, edge j * kBlock + t of a round
// going to thread t, so a load instruction of a wave reads consecutive
// entries of a row.  A thread finds its edges' rows by searching the offsets,
// and hands the four column positions (-1: none) and owners to `edges`, which
// issues every memory trip of a round for all four before using the first
// result.  Replaces ExpandByCta / ExpandByWarp / ExpandByScan
// (b40c/graph/bfs/two_phase/expand_atomic/cta.cuh:215-423).
// Called by every thread; `edges` is called workgroup-converged, and
// `begin` once before, with the tile's edge count.  Edge j of a call is edge
// x0 + j * kBlock of the tile.
//
// A level is bound by its chain of dependent memory trips, not by bytes: one
// row per thread gathered 64 edges a wave at a time made the
// 4318-vertex level of a 100 k-vertex random graph a chain of 16 such rounds
// on nine workgroups, 76 us; spread over the grid it is one round.
// ---------------------------------------------------------------------------
// A tile of more than hub.heavy edges sends its rows from hub.heavy_row edges
// on to the grid tier as well.  The first workgroups to claim anything in a
// level claim its high-degree vertices (an edge leads to a vertex in
// proportion to its degree), and with 2048 items a tile they kept the
// 24.9 M-edge contract-expand step of an R-MAT scale 20 search busy for
// 1200 us while the rest waited.  In a step of one tile per workgroup the
// others have nothing else to do, so there two rounds' edges are heavy.
constexpr int kHeavyTile = 1 << 15, kHeavyTileNarrow = 2 * 4 * kBlock;
constexpr int kHeavyRow = 512, kHeavyRowNarrow = 256;

template <int K, typename Begin, typename Edges>
__device__ __forceinline__ void gather_tile(const int (&beg)[K], int (&end)[K], const int (&par)[K],
                                            const HubList &hub, RowTable &rt, Begin &&begin, Edges &&edges)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    int *tbeg = &rt.beg[0][0], *toff = &rt.excl[0][0], *tpar = &rt.par[0][0];
    int rpos, epos, rtotal, etotal;
    HubList h = hub;
    while (true) {
        int rows = 0, degs = 0;
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (publish_hub_row(beg[k], end[k], par[k], h)) end[k] = beg[k];
            rows += end[k] > beg[k] ? 1 : 0;
            degs += end[k] - beg[k];
        }
        // exclusive sums of rows and edges over the workgroup, in one pass
        const int rincl = wave_inclusive_sum(rows), dincl = wave_inclusive_sum(degs);
        if (lane == kWave - 1) {
            rt.scan[wave] = rincl;
            rt.scan2[wave] = dincl;
        }
        __syncthreads();
        rpos = rincl - rows;
        epos = dincl - degs;
        rtotal = etotal = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const int a = rt.scan[w], b = rt.scan2[w];
            if (w < wave) {
                rpos += a;
                epos += b;
            }
            rtotal += a;
            etotal += b;
        }
        if (etotal <= h.heavy || h.grid_t <= h.heavy_row || h.grid_t == 0x7fffffff) break;
        h.grid_t = h.heavy_row;
        __syncthreads();  // the sums are written again
    }
    begin(etotal);
    for (int r0 = 0; r0 < rtotal; r0 += kBlock) {
        int p = rpos - r0, e = epos;
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (end[k] > beg[k]) {
                if (p >= 0 && p < kBlock) {
                    tbeg[p] = beg[k] - e;  // column position of edge x of the tile: tbeg + x
                    toff[p] = e;
                    tpar[p] = par[k];
                } else if (p == kBlock) {
                    rt.end = e;
                }
                p++;
                e += end[k] - beg[k];
            }
        }
        const int nr = min(rtotal - r0, kBlock);
        if (rtotal - r0 <= kBlock && tid == 0) rt.end = etotal;
        __syncthreads();
        const int e_begin = toff[0], e_end = rt.end;
        int top = 1;  // first step of the search: the largest power of two below nr (uniform)
        while (2 * top < nr) top *= 2;
        // (unsigned: the last round of a tile may reach past 2^31)
        for (unsigned b0 = (unsigned) e_begin; b0 < (unsigned) e_end; b0 += 4 * kBlock) {
            int at[4], pv[4], r[4];
#pragma unroll
            for (int j = 0; j < 4; j++) r[j] = 0;
            for (int st = top; st > 0; st >>= 1) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int q = r[j] + st;
                    if (q < nr && (unsigned) toff[q] <= b0 + (unsigned) (j * kBlock + tid)) r[j] = q;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const unsigned x = b0 + (unsigned) (j * kBlock + tid);
                at[j] = x < (unsigned) e_end ? tbeg[r[j]] + (int) x : -1;
                pv[j] = tpar[r[j]];
            }
            edges(at, pv, b0 + (unsigned) tid);
        }
        __syncthreads();  // the table and the sums are written again next
    }
    if (rtotal == 0) __syncthreads();
}

// ---------------------------------------------------------------------------
// Long rows of a bottom-up step: the lanes of mask lm look for the first
// neighbour in the frontier among columns [beg, end) of their rows; returns
// it to them (other lanes, and rows without one: `none`).  The whole wave
// reads 64 neighbours of each of kLongRows rows at a time, so as many chains
// (column, frontier word) run together; a row that is done makes room for the
// next.  in_frontier(u, in) tests kLongRows neighbours per lane (-1: none).
// (One row at a time made these rows most of a first bottom-up level: 8 to 30
// of them per wave, two memory trips each.)
// ---------------------------------------------------------------------------
constexpr int kLongRows = 4;

template <typename Test>
__device__ __forceinline__ int scan_long_rows(uint64_t lm, int beg, int end, int none, const int *col, Test &&in_frontier)
{
    const int lane = lane_id();
    int found = none;
    int row[kLongRows], at[kLongRows], stop[kLongRows];  // wave-uniform; row: the lane, -1 none
#pragma unroll
    for (int q = 0; q < kLongRows; q++) row[q] = -1;
    while (true) {
        bool any = false;
#pragma unroll
        for (int q = 0; q < kLongRows; q++) {
            if (row[q] < 0 && lm) {
                row[q] = uniform(__builtin_ctzll(lm));
                lm &= lm - 1;
                at[q] = readlane(beg, row[q]);
                stop[q] = readlane(end, row[q]);
            }
            any = any || row[q] >= 0;
        }
        if (!any) return found;
        int u[kLongRows];
        bool in[kLongRows];
#pragma unroll
        for (int q = 0; q < kLongRows; q++) u[q] = row[q] >= 0 && at[q] + lane < stop[q] ? col[at[q] + lane] : -1;
        in_frontier(u, in);
#pragma unroll
        for (int q = 0; q < kLongRows; q++) {
            if (row[q] < 0) continue;
            const uint64_t hm = ballot(in[q]);
            if (hm) {  // (the first in row order)
                const int hit = readlane(u[q], uniform(__builtin_ctzll(hm)));
                if (lane == row[q]) found = hit;
                row[q] = -1;
            } else {
                at[q] += kWave;
                if (at[q] >= stop[q]) row[q] = -1;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Grid barrier for cooperatively launched (co-resident) grids.
// Two-level arrival: workgroup b arrives on leaf counter b % kBarrierFanIn;
// the last arrival at a leaf arrives at the root; the last root arrival
// resets the counters and publishes the new generation into every leaf's
// release word, so waiting workgroups poll kBarrierFanIn different lines
// instead of one.
//
// Memory ordering of a full barrier costs one agent-scope release fence (L2
// write-back) and one acquire fence (L1/L2 invalidate) per workgroup, issued
// by thread 0 around the workgroup barriers.  Polling uses relaxed loads: an acquire load inside
// the spin would invalidate the caches on every poll and slow every other
// workgroup still working.  The last arrivers chain acquire/release fences so
// every workgroup's pre-barrier writes happen-before every post-barrier read.
// Replaces util::GlobalBarrier (b40c/util/global_barrier.cuh:80-126).
// ---------------------------------------------------------------------------
// Every wave drains its own outstanding memory operations first:
// __syncthreads() alone does not wait for other waves' stores, and the
// single write-back of thread 0's release fence must find all of this
// workgroup's stores already in L2, or a store still in flight stays dirty
// in this XCD's L2 and readers elsewhere see old memory.
__device__ __forceinline__ void drain() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

// Release and acquire of the whole caches, by thread 0 for its workgroup
// (every thread of the workgroup calls them).
__device__ __forceinline__ void release_caches()
{
    drain();
    __syncthreads();
    if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
}
__device__ __forceinline__ void refresh_caches()
{
    if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
}

// MAINTAIN: plain stores before the barrier are visible to plain loads after
// it, at the price of a write-back and an invalidate of the XCD's L2 per
// workgroup.  Without it (light barriers) the barrier orders only what goes
// past the XCDs' L2s by itself -- agent- and system-scope loads, stores and
// atomics: a workgroup's have completed before it arrives.  At 256 workgroups
// the maintenance is two thirds of the barrier (6.4 us with, 2.3 without).
// The counter protocol is the same; each of its stores is waited for before
// the store or atomic that may release someone who depends on it.
template <bool MAINTAIN>
__device__ __forceinline__ void grid_barrier_t(Control *ctl)
{
    const unsigned nblocks = gridDim.x;
    const unsigned leaf = blockIdx.x % kBarrierFanIn;
    const unsigned leaves = nblocks < (unsigned) kBarrierFanIn ? nblocks : (unsigned) kBarrierFanIn;
    // workgroups on this leaf: ceil((nblocks - leaf) / fan_in)
    const unsigned leaf_size = (nblocks - leaf + kBarrierFanIn - 1) / kBarrierFanIn;
    drain();
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned *release = &ctl->bar_release[leaf * 32];
        // The generation comes from the one global word, which only the last
        // arriver of a barrier advances (after every workgroup has read it
        // here); waiters then wait for their leaf word to reach gen + 1.
        // Leaf words of leaves a smaller earlier grid never used may lag:
        // they are compared with gen + 1, never with each other.
        const unsigned gen = __hip_atomic_load(&ctl->bar_gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (the generation must be read before this arrival)
        if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        drain();
        unsigned *lc = &ctl->bar_leaf[leaf * 32];
        unsigned arrived = __hip_atomic_fetch_add(lc, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool last = false;
        if (arrived == leaf_size - 1) {
            if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
            __hip_atomic_store(lc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // Relaxed stores to different lines may land in any order, and a
            // relaxed RMW does not wait for them: the reset must be visible
            // before the root arrival that can release this leaf's
            // workgroups, or their next arrival could be overwritten by it.
            if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            drain();
            unsigned r = __hip_atomic_fetch_add(&ctl->bar_root, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (r == leaves - 1) {
                if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
                __hip_atomic_store(&ctl->bar_root, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&ctl->bar_gen, gen + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // the new generation and the root reset before any release
                // word: a released workgroup reads bar_gen at its next
                // barrier, and an old value there would let it straight
                // through
                if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                drain();
                for (unsigned l = 0; l < leaves; l++)
                    __hip_atomic_store(&ctl->bar_release[l * 32], gen + 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                last = true;
            }
        }
        if (!last) {
            while (__hip_atomic_load(release, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gen + 1)
                __builtin_amdgcn_s_sleep(MAINTAIN ? 2 : 1);
        }
        if (MAINTAIN) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}

__device__ __forceinline__ void grid_barrier(Control *ctl) { grid_barrier_t<true>(ctl); }
__device__ __forceinline__ void grid_barrier_light(Control *ctl) { grid_barrier_t<false>(ctl); }

// Thread 0 of block 0 only: waits until every other workgroup has arrived at
// the grid barrier in progress (block 0 itself has not), i.e. until every
// other workgroup is done with whatever it did before that barrier.  Block
// 0's leaf then holds all its workgroups but block 0 and the root all leaves
// but that one; neither count can move on before block 0 arrives, so the wait
// ends exactly once they are reached.
__device__ __forceinline__ void wait_other_arrivals(Control *ctl)
{
    const unsigned nblocks = gridDim.x;
    const unsigned leaves = nblocks < (unsigned) kBarrierFanIn ? nblocks : (unsigned) kBarrierFanIn;
    const unsigned leaf_size = (nblocks + kBarrierFanIn - 1) / kBarrierFanIn;  // of leaf 0
    while (__hip_atomic_load(&ctl->bar_root, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != leaves - 1 ||
           __hip_atomic_load(&ctl->bar_leaf[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != leaf_size - 1)
        __builtin_amdgcn_s_sleep(2);
}

}  // inline namespace (workgroup size)
}  // namespace b40c_hip
