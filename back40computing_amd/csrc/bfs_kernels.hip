// bfs_kernels.hip -- gfx950 breadth-first-search kernels.
//
// One step of the level loop maps a frontier queue to the next one.  The
// step bodies are:
//   expand-contract  vertex frontier -> gather neighbours -> claim -> vertex
//                    frontier (b40c/graph/bfs/expand_contract_atomic/cta.cuh:665-788)
//   contract-expand  edge frontier -> claim -> gather neighbours -> edge
//                    frontier (b40c/graph/bfs/contract_expand_atomic/cta.cuh:573-709)
//   contract         edge frontier -> claim -> vertex frontier
//                    (b40c/graph/bfs/two_phase/contract_atomic/cta.cuh:494-572)
//   expand           vertex frontier -> gather -> edge frontier
//                    (b40c/graph/bfs/two_phase/expand_atomic/cta.cuh:606-719)
//   filter           edge frontier -> visited-bitmask cull -> edge frontier
//                    (b40c/graph/bfs/two_phase/filter_atomic/cta.cuh:308-388)
// Gathering steps have two sub-phases: the tile phase (frontier tiles taken
// by workgroups, their rows' edges spread over the workgroup)
// and, when some rows were long enough for the grid tier, the hub phase in
// which every workgroup takes fixed-size chunks of those rows.
// Each step runs either inside a persistent, cooperatively launched loop with
// in-kernel grid barriers (the reference's KernelGlobalBarrier kernels) or
// as kernel launches per step.
#include "b40c_primitives.hpp"
#include "bfs_device.hpp"
#include "bfs_internal.hpp"

#include <algorithm>
#include <atomic>

namespace b40c_hip {

template <bool PRED>
__device__ __forceinline__ void init_lds(Lds<PRED> &lds)
{
    for (int i = threadIdx.x; i < kHistory; i += kBlock) lds.hist[i] = -1;
    if (threadIdx.x == 0) lds.solo = 0;
    __syncthreads();
}

// Dynamic work assignment: one agent-scope atomic per tile (or chunk).
template <bool PRED>
__device__ __forceinline__ unsigned next_item(unsigned *counter, Lds<PRED> &lds, unsigned k = 1u)
{
    __syncthreads();
    if (threadIdx.x == 0) lds.tile = add_agent(counter, k);
    __syncthreads();
    return lds.tile;
}

// Guided grabs of tiles: one counter atomic hands a workgroup `grab`
// consecutive tiles, about eight grabs per workgroup when a phase has many
// tiles, so the single counter address (whose device-scope atomics
// serialise) stays off the critical path of large levels.
// A phase whose items fit one tile per workgroup and that every workgroup
// runs needs no counter: workgroup b takes tile b (grab 0), and the two round
// trips of the counter atomics (the grab, and the one that finds nothing
// left) leave the level's critical path.  Its tiles are as narrow as spreads
// the items over `want` workgroups.  A workgroup running a step alone
// (lds.solo) grabs every tile itself.
struct TileGrab {
    unsigned next, end, grab, tiles;
    unsigned width;  // items per tile

    // Item i of tile t when tiles are dealt the queue in runs of 16 entries
    // (64 bytes): run k of the tile is the queue's run k * tiles + t.  The
    // members a step claims first, where its output begins, are the
    // high-degree ones; tiles of consecutive members left the first few
    // with most of the edges (R-MAT scale 20, 437602 members, 24.9 M edges:
    // waves lived a quarter of the expansion's 461 us on average).
    __device__ __forceinline__ unsigned dealt(unsigned t, unsigned i) const
    {
        return (((i >> 4) * tiles + t) << 4) + (i & 15u);
    }
};

// tiles per counter atomic of a dynamic assignment
__device__ __forceinline__ unsigned tile_grab_size(const SearchArgs &s, unsigned tiles)
{
    return max(1u, min((unsigned) s.grab_max, tiles / (gridDim.x * 8u)));
}

// Tiles of at most max_width items over n > 0 items.
template <bool PRED>
__device__ __forceinline__ TileGrab tile_grab(const SearchArgs &s, unsigned n, const Lds<PRED> &lds,
                                              unsigned max_width, unsigned want)
{
    if (!lds.solo && n <= gridDim.x * max_width) {
        const unsigned wgs = max(min(want, gridDim.x), (n + max_width - 1) / max_width);
        const unsigned width = min(((n + wgs - 1) / wgs + 15u) & ~15u, max_width);
        const unsigned tiles = (n + width - 1) / width;
        return TileGrab{blockIdx.x, blockIdx.x < tiles ? blockIdx.x + 1 : blockIdx.x, 0u, tiles, width};
    }
    const unsigned tiles = (n + max_width - 1) / max_width;
    return TileGrab{0u, 0u, tile_grab_size(s, tiles), tiles, max_width};
}

// Next tile index of the workgroup (workgroup-uniform); with a static
// assignment, the phase's tile count once the workgroup's tile is done.
template <bool PRED>
__device__ __forceinline__ unsigned next_tile(unsigned *counter, Lds<PRED> &lds, TileGrab &tg)
{
    if (tg.grab == 0) {
        __syncthreads();  // the LDS reuse fence of a grab
        return tg.next == tg.end ? tg.tiles : tg.next++;
    }
    if (tg.next == tg.end) {
        tg.next = next_item(counter, lds, tg.grab);
        tg.end = tg.next + tg.grab;
    } else {
        __syncthreads();  // same LDS reuse fence as a fresh grab
    }
    return tg.next++;
}

// LDS history hash: true if u may be new to this workgroup.  A hit means
// another lane of this workgroup already took u through the claim, so this
// copy can be dropped without touching global memory.  Racing lanes may both
// miss; the claim that follows settles them.  Cf. HistoryCull / WarpCull
// (b40c/graph/bfs/two_phase/contract_atomic/cta.cuh:276-327).
template <bool PRED>
__device__ __forceinline__ bool history_pass(Lds<PRED> &lds, int u)
{
    unsigned h = ((unsigned) u * 0x9E3779B1u) >> (32 - 10);
    static_assert(kHistory == 1024, "history hash uses 10 bits");
    if (lds.hist[h] == u) return false;
    lds.hist[h] = u;
    return true;
}

// How a grid-wide step meets the caches around it (grid-uniform):
// light: a light barrier follows, so what other workgroups read next goes
//   past the XCD's L2 (queue entries); the step is small, and reads the rows
//   of its candidates before their claims have answered;
// stale: a light barrier came before, so this XCD's L2 may hold visited words
//   from before other workgroups' claims: pre-reads go past it.  (A word that
//   is too old only costs a claim that fails, but on a lattice every second
//   edge leads back to a vertex visited a level or two before.)
// launched: the step is a launch of its own, whose hub launch follows anyway.
struct StepIo {
    bool light, stale, launched = false;
};

template <bool PRED>
__device__ __forceinline__ WaveQueue<PRED> make_queue(const SearchArgs &s, int step, Lds<PRED> &lds,
                                                      bool through = false)
{
    const int wave = threadIdx.x / kWave;
    WaveQueue<PRED> wq;
    wq.buf = lds.wq[wave];
    if constexpr (PRED) wq.pbuf = lds.wqp.buf[wave];
    else wq.pbuf = nullptr;
    wq.count = 0;
    wq.through = through;
    wq.out = s.q[(step + 1) & 1];
    wq.pout = PRED ? s.pq[(step + 1) & 1] : nullptr;
    wq.out_len = &s.ctl->qlen[(step + 1) % 3];
    wq.cap = s.cap;
    wq.overflow = &s.ctl->overflow;
    wq.overflow_step = &s.ctl->ovf[(step + 1) % 3];
    return wq;
}

// Steps of at most one kBlock-item tile per workgroup: rows of a grid-tier
// chunk and more go to the grid tier, so that no workgroup of such a short
// step strides a long row alone.  Grid-uniform (n is read after a barrier).
__device__ __forceinline__ bool narrow_step(unsigned n) { return (n + kBlock - 1) / kBlock <= gridDim.x; }

// Grid-tier list of a gathering step over n input items.
__device__ __forceinline__ HubList hub_list(const SearchArgs &s, int step, bool enabled, unsigned n)
{
    HubList h;
    h.entries = s.hubs[step & 1];
    h.cap = s.hub_cap;
    h.alloc = &s.ctl->hub_alloc[step & 1];
    h.grid_t = enabled ? s.grid_t : 0x7fffffff;
    if (enabled && narrow_step(n)) h.grid_t = min(h.grid_t, kHubChunk);
    h.tag = 0;
    h.out_len = nullptr;
    h.heavy = narrow_step(n) ? kHeavyTileNarrow : kHeavyTile;
    h.heavy_row = narrow_step(n) ? kHeavyRowNarrow : kHeavyRow;
    return h;
}

// End of a step for the whole workgroup (every thread calls it): the waves'
// staged queue entries are reserved with one atomic, and their degree sums
// are folded into one update.  256 workgroups' atomics on one address cost a
// level about 2 us (8 ns each) on top of its barrier and plain stores to one
// address 6 us, so a step keeps to these two: the deepest label is noted by
// one workgroup at the top of the next step (prepare_step), and the visited
// edges are summed by whoever decides on them.
//
// `uncounted` (per lane) adds frontier members that are not staged in the
// queue: a bottom-up level records its output only in the frontier bitmap,
// and the queue length alone carries its size.
// `labeled` (per lane; contract-expand): labelled vertices with depth
// `depth`, to be noted here if the workgroup stages no output at all.
template <bool PRED>
__device__ void finish_step(WaveQueue<PRED> &wq, Lds<PRED> &lds, Control *ctl, int step, unsigned fe, bool track,
                            int uncounted = 0, bool labeled = false, int depth = -1)
{
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int lo = wave_inclusive_sum((int) (fe & 0xFFFFu));
    int hi = wave_inclusive_sum((int) (fe >> 16));
    int extra = wave_inclusive_sum(uncounted);
    bool any = ballot(labeled) != 0;
    if (lane == kWave - 1) {  // the inclusive sums end in the last lane
        lds.ep_count[wave] = (unsigned) wq.count;
        lds.ep_extra[wave] = (unsigned) extra;
        lds.ep_fe[wave] = ((unsigned long long) (unsigned) hi << 16) + (unsigned long long) (unsigned) lo;
        lds.ep_lab[wave] = any ? 1 : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned tot = 0, ext = 0;
        unsigned long long fsum = 0;
        int lab = 0;
        for (int w = 0; w < kWaves; w++) {
            tot += lds.ep_count[w];
            ext += lds.ep_extra[w];
            fsum += lds.ep_fe[w];
            lab |= lds.ep_lab[w];
        }
        lds.ep_base = (tot | ext) ? add_agent(wq.out_len, tot + ext) : 0u;
        if (track && fsum)
            __hip_atomic_fetch_add(&ctl->fedges[(step + 1) % 3], fsum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (lab && tot == 0) atomicMax(&ctl->max_depth, depth);
    }
    __syncthreads();
    unsigned off = lds.ep_base;
    for (int w = 0; w < wave; w++) off += lds.ep_count[w];
    const unsigned cnt = (unsigned) wq.count;
    const unsigned lim = off < wq.cap ? min(cnt, wq.cap - off) : 0u;
    if (lim < cnt && lane == 0) {
        st_agent(wq.overflow, 1u);
        st_agent(wq.overflow_step, 1u);
    }
    for (unsigned i = (unsigned) lane; i < lim; i += kWave) wq.store(off + i, wq.buf[i], PRED ? wq.pbuf[i] : -1);
    wq.count = 0;
}

__device__ __forceinline__ unsigned long long ld64_agent(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Generic phases
// ---------------------------------------------------------------------------

// Hub phase: every workgroup takes kHubChunk-edge chunks of the rows that
// the tile phase published, until all chunks are done.  Must follow a grid
// barrier (or kernel boundary) after the tile phase.  run_chunk(b, e, par)
// consumes columns [b, e) of a row of par.
template <bool PRED, typename Chunk>
__device__ __forceinline__ void hub_phase_chunks(const SearchArgs &s, Cursor c, Lds<PRED> &lds, Chunk &&run_chunk)
{
    unsigned long long a = __hip_atomic_load(&s.ctl->hub_alloc[c.step & 1], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    unsigned entries = (unsigned) (a >> 32);
    if (entries > s.hub_cap) entries = s.hub_cap;
    if (entries == 0) return;
    const HubEntry *list = s.hubs[c.step & 1];
    HubEntry lastent = list[entries - 1];
    constexpr int chunk = kHubChunk;
    unsigned total = lastent.first_chunk + (unsigned) ((lastent.end - lastent.beg + chunk - 1) / chunk);
    // guided grabs of consecutive chunks, as for tiles: a level of many hub
    // chunks must not queue on the one chunk counter
    TileGrab tg{0u, 0u, max(1u, min((unsigned) s.grab_max, total / (gridDim.x * 8u))), 0u, 1u};
    unsigned hint = 0;  // thread 0: entry of this workgroup's previous chunk
    while (true) {
        unsigned ch = next_tile(&s.ctl->hub_steal[c.step & 1], lds, tg);
        if (ch >= total) break;
        if (threadIdx.x == 0) {
            const unsigned lo = hub_entry_of(list, entries, ch, hint);
            hint = lo;
            HubEntry e = list[lo];
            int b = e.beg + (int) (ch - e.first_chunk) * chunk;
            lds.cta_beg = b;
            lds.cta_end = min(e.end, b + chunk);
            lds.cta_par = e.par;
            lds.cta_out = (unsigned) e.tag + (unsigned) (b - e.beg);
        }
        __syncthreads();
        run_chunk(lds.cta_beg, lds.cta_end, lds.cta_par);
    }
}


// The same with gather_tile's edge consumer (four column positions per
// thread and round).
template <bool PRED, typename Edges>
__device__ __forceinline__ void hub_phase(const SearchArgs &s, Cursor c, Lds<PRED> &lds, Edges &&edges)
{
    hub_phase_chunks<PRED>(s, c, lds, [&](int b, int e, int par) {
        for (int k = b; k < e; k += 4 * kBlock) {
            int at[4], pv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int x = k + j * kBlock + (int) threadIdx.x;
                at[j] = x < e ? x : -1;
                pv[j] = par;
            }
            edges(at, pv, 0u);
        }
    });
}

// Claims of one thread's edge slots: at[k] = column position of slot k (or
// -1), pv[k] = its row's owner.  Claims the unvisited neighbours, labels
// them, and returns the mask of the slots k that claimed u[k] (row
// [ub[k], ud[k])).  Each memory trip (column entry, visited word, claim,
// row bounds) is issued for every slot before the first result is used.
//
// LOCAL: the calling workgroup is the only one touching the labels and the
// visited words (block 0's fast path, between two grid barriers).  Its
// claims are then workgroup-scope atomics, done in this XCD's L2, where
// agent-scope ones must be coherent across the eight XCDs; the barrier
// before the path invalidated stale lines, and the one after it writes the
// path's lines back.  Column entries are read through the caches: the next
// level's rows sit next to this level's on a lattice.  With vbits (LOCAL
// only) the claims are LDS atomics on the path's copy of the visited
// bitmap: no pre-read and no memory trip between a column entry and the
// claimed vertex's row bounds.
// Without ROWS the row bounds are not read (the caller does not gather).
// The claims are atomic whatever the cull mode: with four edges per thread in
// flight, racing plain stores (claim_best_effort) passed so many duplicates
// that queues of four times the vertices overflowed.  EXACT says that no step
// of the search claims otherwise (only best-effort chained contractions do,
// chained_step), so that every labelled vertex has its visited bit.
// fast_claim_vertices: the same for vertices u[k] (-1: none) already at hand.
template <bool PRED, bool EXACT, bool LOCAL, int S, bool ROWS = true>
__device__ __forceinline__ unsigned fast_claim_vertices(const GraphArgs &g, const SearchArgs &s, int next_depth,
                                                        const int (&pv)[S], const int (&u)[S], int (&ub)[S],
                                                        int (&ud)[S], bool ldsv, unsigned *vbits,
                                                        StepIo io = StepIo{false, false})
{
    unsigned old[S];
    const bool coherent = s.coherent_filter || (!LOCAL && io.stale);
    // light steps: the candidates' rows, read beside their claims
    int rb[S], rd[S];
    if (LOCAL && ldsv) {
#pragma unroll
        for (int k = 0; k < S; k++) {
            old[k] = ~0u;
            if (u[k] >= 0)
                old[k] = __hip_atomic_fetch_or(vbits + (u[k] >> 5), 1u << (u[k] & 31), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    } else {
        // visited words (a set bit is final), then claims of the clear ones
        unsigned cur[S];
#pragma unroll
        for (int k = 0; k < S; k++) {
            cur[k] = ~0u;
            if (u[k] >= 0) {
                unsigned *w = s.visited + (u[k] >> 5);
                cur[k] = coherent ? __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *w;
            }
        }
        // The claims' results are read only after all are issued (a use
        // next to its atomic would wait out each round trip in turn).
#pragma unroll
        for (int k = 0; k < S; k++) {
            old[k] = ~0u;
            const unsigned bit = 1u << (u[k] & 31);
            if (u[k] >= 0 && !(cur[k] & bit)) {
                // agent scope unless LOCAL: other workgroups claim
                // concurrently, and another XCD's L2 may hold this word from
                // before an earlier step's claims
                if (LOCAL)
                    old[k] = __hip_atomic_fetch_or(s.visited + (u[k] >> 5), bit, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                else
                    old[k] = __hip_atomic_fetch_or(s.visited + (u[k] >> 5), bit, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if constexpr (!LOCAL && ROWS) {
            if (io.light) {
#pragma unroll
                for (int k = 0; k < S; k++) {
                    rb[k] = 0;
                    rd[k] = 0;
                    if (u[k] >= 0 && !((cur[k] >> (u[k] & 31)) & 1u)) {
                        rb[k] = g.row[u[k]];
                        rd[k] = g.row[u[k] + 1];
                    }
                }
            }
        }
    }
    // (the empty asm keeps the compiler from folding a use into the
    // atomic's own block)
#pragma unroll
    for (int k = 0; k < S; k++) asm volatile("" : "+v"(old[k]));
    unsigned fresh = 0;
#pragma unroll
    for (int k = 0; k < S; k++)
        if (!((old[k] >> (u[k] & 31)) & 1u)) fresh |= 1u << k;
    if (!EXACT) {
        // chained contractions may have lost bits of labelled vertices
        int dep[S];
#pragma unroll
        for (int k = 0; k < S; k++) dep[k] = ((fresh >> k) & 1) ? s.depth[u[k]] : -1;
#pragma unroll
        for (int k = 0; k < S; k++)
            if (dep[k] != -1) fresh &= ~(1u << k);
    }
#pragma unroll
    for (int k = 0; k < S; k++) {
        ub[k] = 0;
        ud[k] = 0;
        if ((fresh >> k) & 1) {
            s.depth[u[k]] = next_depth;
            if (PRED) s.pred[u[k]] = pv[k];
            if (!LOCAL && io.light) {
                if (ROWS) {
                    ub[k] = rb[k];
                    ud[k] = rd[k];
                }
            } else if (ROWS) {
                ub[k] = g.row[u[k]];
                ud[k] = g.row[u[k] + 1];
            }
        }
    }
    return fresh;
}

template <bool PRED, bool EXACT, bool LOCAL, int S>
__device__ __forceinline__ unsigned fast_claim_slots(const GraphArgs &g, const SearchArgs &s, int next_depth,
                                                     const int (&at)[S], const int (&pv)[S], int (&u)[S],
                                                     int (&ub)[S], int (&ud)[S], bool ldsv = false,
                                                     unsigned *vbits = nullptr, StepIo io = StepIo{false, false})
{
#pragma unroll
    for (int k = 0; k < S; k++)
        u[k] = at[k] < 0 ? -1 : LOCAL ? g.col[at[k]] : __builtin_nontemporal_load(g.col + at[k]);
    return fast_claim_vertices<PRED, EXACT, LOCAL, S>(g, s, next_depth, pv, u, ub, ud, ldsv, vbits, io);
}

// Workgroups worth running a top-down step of `fe` frontier edges: about
// 1024 edges each (two per thread), fewer workgroups than that leave a
// longer chain, more only add reservation atomics.
__device__ __forceinline__ unsigned edge_workgroups(unsigned long long fe)
{
    return (unsigned) min(fe / 1024ull + 1ull, (unsigned long long) gridDim.x);
}

// ---------------------------------------------------------------------------
// Step bodies.  All threads of the workgroup execute them together.
// sub == 0 runs the tile phase, sub == 1 the hub phase.  The bodies and the
// level loop's other parts are force-inlined: one left out of line takes the
// kernel's argument structs by address, and the compiler then copies them to
// scratch and reads every field from there for the whole kernel.
// ---------------------------------------------------------------------------
// (fe_in: the step's frontier edges)
template <bool PRED>
__device__ __forceinline__ void body_expand_contract(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds,
                                     int sub, bool hubs, unsigned long long fe_in, StepIo io,
                                     unsigned *next_bits = nullptr, bool from_bitmap = false)
{
    WaveQueue<PRED> wq = make_queue<PRED>(s, c.step, lds, io.light);
    const int *in = s.q[c.step & 1];
    const int next_depth = c.iteration + 1;
    unsigned fe = 0;
    auto begin = [](int) {};
    auto edges = [&](const int (&at)[4], const int (&pv)[4], unsigned) {
        int u[4], ub[4], ud[4];
        const unsigned fresh =
            fast_claim_slots<PRED, true, false, 4>(g, s, next_depth, at, pv, u, ub, ud, false, nullptr, io);
#pragma unroll
        for (int j = 0; j < 4; j++) fe += (unsigned) (ud[j] - ub[j]);
        // a clear frontier bitmap becomes the next frontier's, exactly
        if (next_bits) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if ((fresh >> j) & 1)
                    __hip_atomic_fetch_or(next_bits + (u[j] >> 5), 1u << (u[j] & 31), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) wq.push((fresh >> j) & 1, u[j], pv[j]);
    };
    if (sub == 0 && from_bitmap) {
        // The frontier is frontier bitmap fbm[c.iteration & 1], as a
        // bottom-up level left it: each workgroup takes kBlock-word tiles
        // of it, clears them and the other bitmap's words (so both are
        // clear after the step, as a top-down level needs them), and
        // gathers up to two members per thread per round.
        const HubList hub = hub_list(s, c.step, hubs, n);
        unsigned *bm = s.fbm[c.iteration & 1];
        unsigned *other = s.fbm[(c.iteration + 1) & 1];
        const unsigned words = ((unsigned) g.nodes + 31) >> 5;
        for (unsigned w0 = blockIdx.x * kBlock; w0 < words; w0 += gridDim.x * kBlock) {
            const unsigned w = w0 + threadIdx.x;
            unsigned bits = 0u;
            if (w < words) {
                bits = bm[w];
                bm[w] = 0u;
                other[w] = 0u;
            }
            while (__syncthreads_or(bits != 0u)) {
                int beg[2] = {0, 0}, end[2] = {0, 0}, par[2] = {-1, -1};
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    if (bits) {
                        par[k] = (int) ((w << 5) + (unsigned) __builtin_ctz(bits));
                        bits &= bits - 1u;
                    }
                }
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    if (par[k] >= 0) {
                        beg[k] = g.row[par[k]];
                        end[k] = g.row[par[k] + 1];
                    }
                }
                gather_tile<2>(beg, end, par, hub, lds.rt, begin, edges);
            }
        }
    } else if (sub == 0) {
        HubList hub = hub_list(s, c.step, hubs, n);
        // The few members of a launched step lie on a workgroup or two, and
        // its hub launch follows anyway: rows of a wave and more go there
        // (R-MAT scale 20, a level of 10 members and 73 k new vertices: 60
        // us with rows of 2048 alone, 48 from 64 on, 50 from 256 and 512).
        if (io.launched && n < (unsigned) kBlock) hub.grid_t = min(hub.grid_t, kWave);
        TileGrab tg = tile_grab(s, n, lds, kBlock, edge_workgroups(fe_in));
        while (true) {
            const unsigned t = next_tile(&s.ctl->steal[c.step & 1], lds, tg);
            if (t >= tg.tiles) break;
            const unsigned i = tg.dealt(t, threadIdx.x);
            int beg[1] = {0}, end[1] = {0}, par[1] = {-1};
            if (threadIdx.x < tg.width && i < n) {
                par[0] = ld_queue(in + i);
                beg[0] = g.row[par[0]];
                end[0] = g.row[par[0] + 1];
            }
            gather_tile<1>(beg, end, par, hub, lds.rt, begin, edges);
        }
    } else {
        hub_phase<PRED>(s, c, lds, edges);
    }
    finish_step<PRED>(wq, lds, s.ctl, c.step, fe, s.track_edges != 0);
}

// Bottom-up step of a direction-optimizing search (Beamer, Asanovic,
// Patterson, "Direction-Optimizing Breadth-First Search", SC'12): every
// unvisited vertex scans its row for a neighbour in the current frontier
// bitmap fbm[d & 1] and stops at the first one (in row order).
//
// The level is bound by each wave's chain of dependent loads (row bounds,
// neighbours, frontier words), not by bytes.  Each wave owns one contiguous
// run of 64-vertex groups (static partition: no tile counter, no workgroup
// barrier; scrambled ids balance the runs) and walks it in two stages:
//   1. the visited words and row bounds of kBuGroups groups at a time
//      (prefetched one step ahead) give the vertices still to search with a
//      non-empty row; they are queued in the wave's LDS -- on later levels
//      only a few lanes of a group have work;
//   2. every 128 queued vertices are scanned with all lanes busy, two per
//      lane: four neighbours of each per round, all eight loads of a round
//      in flight; rows of kBuLong+ neighbours get one such round and then a
//      wave-wide scan of the rest, several rows at a time (a high-degree
//      vertex usually finds a frontier neighbour among its first four).
// Parents found are collected as bits in LDS per window of kBuWindow groups
// and written once per word: visited |= found, next frontier = found (the
// next-frontier word is overwritten in full, which also clears it).
constexpr int kBuLong = 64;
constexpr int kBuGroups = 2;
constexpr int kBuQueue = 192;   // queued vertices per wave (a two-entry scan and a group more)
constexpr int kBuWindow = 32;   // groups per window of found bits (2 words each)
static_assert(3 * kBuQueue + 2 * kBuWindow <= kWaveQueueCap, "bottom-up LDS use fits the wave's staging area");

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool PRED>
__device__ __forceinline__ void body_bottom_up(const GraphArgs &g, const SearchArgs &s, Cursor c, Lds<PRED> &lds)
{
    WaveQueue<PRED> wq = make_queue<PRED>(s, c.step, lds);
    const unsigned *cur = s.fbm[c.iteration & 1];
    unsigned *nxt = s.fbm[(c.iteration + 1) & 1];
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    const int next_depth = c.iteration + 1;
    const unsigned words = ((unsigned) g.nodes + 31) >> 5;
    unsigned fe = 0;
    int found = 0;
    int *qv = lds.wq[wave];
    int *qb = qv + kBuQueue;
    int *qe = qb + kBuQueue;
    unsigned *fbits = reinterpret_cast<unsigned *>(qe + kBuQueue);

    const unsigned groups = ((unsigned) g.nodes + kWave - 1) / kWave;
    const unsigned nwaves = gridDim.x * kWaves;
    const unsigned gw = blockIdx.x * kWaves + (unsigned) wave;
    const unsigned per = (groups + nwaves - 1) / nwaves;
    const unsigned g_begin = gw * per;
    const unsigned g_end = min(groups, (gw + 1) * per);

    // Scans the first cnt (1..128, wave-uniform) queued vertices of the
    // window whose first visited word is word0: lane l takes entries l and
    // l + 64, whose rounds of four neighbours run with all loads in flight.
    auto scan = [&](int cnt, unsigned word0) {
        int v[2], beg[2], end[2], pos[2], lim[2], parent[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int i = lane + h * kWave;
            v[h] = -1;
            beg[h] = 0;
            end[h] = 0;
            if (i < cnt) {
                v[h] = qv[i];
                beg[h] = qb[i];
                end[h] = qe[i];
            }
            pos[h] = beg[h];
            lim[h] = end[h] - beg[h] < kBuLong ? end[h] : min(end[h], beg[h] + 4);
            parent[h] = -1;
        }
        while ((parent[0] < 0 && pos[0] < lim[0]) || (parent[1] < 0 && pos[1] < lim[1])) {
            int u[8];
            unsigned fw[8];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    u[h * 4 + j] = parent[h] < 0 && pos[h] + j < lim[h] ? g.rcol[pos[h] + j] : -1;
#pragma unroll
            for (int k = 0; k < 8; k++) fw[k] = u[k] >= 0 ? cur[u[k] >> 5] : 0u;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 3; j >= 0; j--)  // the first hit in row order wins
                    if (u[h * 4 + j] >= 0 && ((fw[h * 4 + j] >> (u[h * 4 + j] & 31)) & 1u)) parent[h] = u[h * 4 + j];
            pos[0] += 4;
            pos[1] += 4;
        }
        // rows of kBuLong+ neighbours with no parent among their first four:
        // a wave-wide scan of the rest
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint64_t lm = ballot(parent[h] < 0 && lim[h] < end[h]);
            if (lm)
                parent[h] = scan_long_rows(lm, lim[h], end[h], parent[h], g.rcol,
                                           [&](const int (&u)[kLongRows], bool (&in)[kLongRows]) {
                                               unsigned fw[kLongRows];
#pragma unroll
                                               for (int q = 0; q < kLongRows; q++)
                                                   fw[q] = u[q] >= 0 ? cur[u[q] >> 5] : 0u;
#pragma unroll
                                               for (int q = 0; q < kLongRows; q++)
                                                   in[q] = u[q] >= 0 && ((fw[q] >> (u[q] & 31)) & 1u);
                                           });
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (parent[h] >= 0) {
                s.depth[v[h]] = next_depth;
                if (PRED) s.pred[v[h]] = parent[h];
                fe += (unsigned) (end[h] - beg[h]);
                found++;
                __hip_atomic_fetch_or(&fbits[((unsigned) v[h] >> 5) - word0], 1u << (v[h] & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
    };
    // Moves queue entries [from, from + n) to the front.
    auto shift = [&](int from, int n) {
        int v = 0, b = 0, e = 0;
        if (lane < n) {
            v = qv[from + lane];
            b = qb[from + lane];
            e = qe[from + lane];
        }
        wave_lds_sync();
        if (lane < n) {
            qv[lane] = v;
            qb[lane] = b;
            qe[lane] = e;
        }
        wave_lds_sync();
    };

    unsigned vis_n[kBuGroups];
    int beg_n[kBuGroups], end_n[kBuGroups];
    auto load_groups = [&](unsigned g0, unsigned g_stop) {
#pragma unroll
        for (int k = 0; k < kBuGroups; k++) {
            const int vv = (int) ((g0 + (unsigned) k) * kWave + (unsigned) lane);
            const bool ok = g0 + (unsigned) k < g_stop && vv < g.nodes;
            vis_n[k] = ok ? s.visited[(unsigned) vv >> 5] : ~0u;
            beg_n[k] = ok ? g.rrow[vv] : 0;
            end_n[k] = ok ? g.rrow[vv + 1] : 0;
        }
    };
    if (g_begin < g_end) load_groups(g_begin, g_end);
    for (unsigned w_begin = g_begin; w_begin < g_end; w_begin += kBuWindow) {
        const unsigned w_end = min(g_end, w_begin + kBuWindow);
        const unsigned word0 = 2 * w_begin;
        fbits[lane] = 0u;  // 64 lanes, 2 * kBuWindow words
        wave_lds_sync();
        int qn = 0;
        for (unsigned gi = w_begin; gi < w_end; gi += kBuGroups) {
            unsigned vis[kBuGroups];
            int beg[kBuGroups], end[kBuGroups];
#pragma unroll
            for (int k = 0; k < kBuGroups; k++) {
                vis[k] = vis_n[k];
                beg[k] = beg_n[k];
                end[k] = end_n[k];
            }
            // the next groups of this run (the window boundary does not stop the pipeline)
            if (gi + kBuGroups < g_end) load_groups(gi + kBuGroups, g_end);
            bool todo[kBuGroups];
#pragma unroll
            for (int k = 0; k < kBuGroups; k++) {
                const int v = (int) ((gi + (unsigned) k) * kWave + (unsigned) lane);
                todo[k] = gi + (unsigned) k < w_end && v < g.nodes && ((vis[k] >> (v & 31)) & 1u) == 0 &&
                          end[k] > beg[k];
            }
#pragma unroll
            for (int k = 0; k < kBuGroups; k++) {
                const uint64_t m = ballot(todo[k]);
                if (todo[k]) {
                    const int p = qn + lanes_below(m);
                    qv[p] = (int) ((gi + (unsigned) k) * kWave + (unsigned) lane);
                    qb[p] = beg[k];
                    qe[p] = end[k];
                }
                qn += __popcll(m);
                if (qn >= 2 * kWave) {
                    wave_lds_sync();
                    scan(2 * kWave, word0);
                    shift(2 * kWave, qn - 2 * kWave);
                    qn -= 2 * kWave;
                }
            }
        }
        wave_lds_sync();
        while (qn > 0) {
            const int cnt = min(qn, 2 * kWave);
            scan(cnt, word0);
            if (qn > cnt) shift(cnt, qn - cnt);
            qn -= cnt;
        }
        wave_lds_sync();
        // the window's visited and next-frontier words (the wave owns them)
        const unsigned w = word0 + (unsigned) lane;
        if (lane < 2 * (int) (w_end - w_begin) && w < words) {
            const unsigned bits = fbits[lane];
            if (bits) s.visited[w] |= bits;
            nxt[w] = bits;
        }
        wave_lds_sync();
    }
    // The level's output is the bitmap nxt; only its size goes to the queue
    // length (queue_from_bitmap materialises the queue if the search turns
    // top-down again).
    finish_step<PRED>(wq, lds, s.ctl, c.step, fe, true, found);
}

// Writes the members of frontier bitmap fbm[c.iteration & 1] into the input
// queue of step c (a bottom-up level records its output only as a bitmap),
// clearing both frontier bitmaps on the way.
// Grid-wide; a grid barrier or kernel boundary must follow before the queue
// is read.  Reservations come from ctl->compact, which the previous step
// zeroed.
template <bool PRED>
__device__ __forceinline__ void queue_from_bitmap(const GraphArgs &g, const SearchArgs &s, Cursor c, Lds<PRED> &lds)
{
    unsigned *bm = s.fbm[c.iteration & 1];
    unsigned *other = s.fbm[(c.iteration + 1) & 1];
    int *out = s.q[c.step & 1];
    const unsigned words = ((unsigned) g.nodes + 31) >> 5;
    const unsigned stride = gridDim.x * kBlock;
    for (unsigned w0 = blockIdx.x * kBlock; w0 < words; w0 += stride) {
        const unsigned w = w0 + threadIdx.x;
        const unsigned bits = w < words ? bm[w] : 0u;
        // top-down levels leave both bitmaps clear (see frontier_bitmap_pass)
        if (w < words) {
            bm[w] = 0u;
            other[w] = 0u;
        }
        int total = 0;
        int excl = block_exclusive_sum(__popc(bits), lds.ep_scan, &total);
        if (threadIdx.x == 0) lds.ep_base = total ? add_agent(&s.ctl->compact, (unsigned) total) : 0u;
        __syncthreads();
        unsigned pos = lds.ep_base + (unsigned) excl;
        for (unsigned b = bits; b; b &= b - 1) {
            if (pos < s.cap) out[pos] = (int) ((w << 5) + (unsigned) __builtin_ctz(b));
            pos++;
        }
        __syncthreads();
    }
}

// Contraction of one tile of an edge frontier: threads take up to kItems
// items each (kBlock apart), cull them through the history hash, and claim
// the rest with every memory trip in flight for all of them.  Returns the
// mask of the items k that claimed u[k] (parent pv[k], row [ub[k], ud[k])).
constexpr int kItems = 4;

template <bool PRED, bool EXACT, bool ROWS>
__device__ __forceinline__ unsigned contract_tile(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n,
                                                  unsigned base, unsigned width, Lds<PRED> &lds, StepIo io,
                                                  int (&u)[kItems], int (&pv)[kItems], int (&ub)[kItems],
                                                  int (&ud)[kItems])
{
    const int *in = s.q[c.step & 1];
    const int *pin = s.pq[c.step & 1];
#pragma unroll
    for (int k = 0; k < kItems; k++) {
        const unsigned o = (unsigned) (k * kBlock) + threadIdx.x;
        const bool ok = o < width && base + o < n;
        u[k] = ok ? ld_queue(in + base + o) : -1;
        pv[k] = PRED && ok ? ld_queue(pin + base + o) : -1;
    }
#pragma unroll
    for (int k = 0; k < kItems; k++)
        if (u[k] >= 0 && !history_pass<PRED>(lds, u[k])) u[k] = -1;
    return fast_claim_vertices<PRED, EXACT, false, kItems, ROWS>(g, s, c.iteration, pv, u, ub, ud, false, nullptr,
                                                                 io);
}

// The rows of a large vertex frontier, waves alone: wave w takes runs w, w + waves, ... of up to 64 queue entries (the
// high-degree members, claimed first, are spread over all of them), and
// nothing but the published rows waits for the workgroup.  Rows of
// kWaveRow edges and more are read a row per load instruction, eight rows
// in flight; shorter ones share load instructions through the wave's edge
// offsets, four of them in flight.  Rows of kWaveHubRow edges and more are
// published: the grid tier follows behind a grid barrier.  `edges` gets the
// neighbours (-1: none) and owners of four or eight edges per lane, called
// wave-converged.  Returns this lane's share of the edges not published.
// (A workgroup's row table, as gather_tile has it, left the waves of a
// bit-marked step in step: 166 us for 437602 rows of 24.9 M edges, about 80
// like this.)
constexpr int kWaveRow = 32, kWaveHubRow = 512;

template <typename Edges>
__device__ __forceinline__ unsigned long long wave_rows(const GraphArgs &g, const int *in, unsigned n,
                                                        const HubList &hub, RowTable &rt, Edges &&edges)
{
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int *excl = rt.excl[wave], *rb = rt.beg[wave], *rp = rt.par[wave];
    unsigned long long met = 0;
    // runs of equal length, as many for every wave
    const unsigned stride = gridDim.x * kWaves;
    const unsigned rounds = (n + stride * kWave - 1) / (stride * kWave);
    const unsigned width = (n + stride * rounds - 1) / (stride * rounds), runs = (n + width - 1) / width;
    unsigned t = (unsigned) wave * gridDim.x + blockIdx.x;
    auto member = [&](unsigned run) {
        const unsigned long long i = (unsigned long long) run * width + (unsigned) lane;
        return (unsigned) lane < width && i < n ? ld_queue(in + i) : -1;
    };
    int v_next = member(t), b_next = 0, e_next = 0;
    if (v_next >= 0) {
        b_next = g.row[v_next];
        e_next = g.row[v_next + 1];
    }
    constexpr int U = 8;  // rows in flight
    for (; t < runs; t += stride) {
        const int v = v_next, beg = b_next;
        int end = e_next;
        v_next = member(t + stride);
        if (publish_hub_row(beg, end, v, hub)) end = beg;
        met += (unsigned long long) (end - beg);
        uint64_t wm = ballot(end - beg >= kWaveRow);
        while (wm) {
            int b[U], e[U], p[U], longest = 0;
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int l = wm ? uniform(__builtin_ctzll(wm)) : 0;
                b[q] = readlane(beg, l);
                e[q] = wm ? readlane(end, l) : b[q];
                p[q] = readlane(v, l);
                wm &= wm - 1;  // (0 stays 0)
                longest = max(longest, e[q] - b[q]);
            }
            for (int k = lane; k - lane < longest; k += kWave) {
                int u[U];
#pragma unroll
                for (int q = 0; q < U; q++) u[q] = k < e[q] - b[q] ? __builtin_nontemporal_load(g.col + b[q] + k) : -1;
                edges(u, p);
            }
        }
        // the next run's row bounds, behind its members
        b_next = e_next = 0;
        if (v_next >= 0) {
            b_next = g.row[v_next];
            e_next = g.row[v_next + 1];
        }
        const int len = end - beg < kWaveRow ? end - beg : 0;
        const int incl = wave_inclusive_sum(len);
        const int total = readlane(incl, kWave - 1);
        if (total == 0) continue;
        excl[lane] = incl - len;
        rb[lane] = beg - (incl - len);
        rp[lane] = v;
        wave_lds_sync();
        for (int r = 0; r < total; r += 4 * kWave) {
            int u[4], p[4], at[4];
#pragma unroll
            for (int q = 0; q < 4; q++) at[q] = 0;
#pragma unroll
            for (int st = 32; st > 0; st >>= 1) {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (excl[at[q] + st] <= r + q * kWave + lane) at[q] += st;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int x = r + q * kWave + lane;
                u[q] = x < total ? __builtin_nontemporal_load(g.col + rb[at[q]] + x) : -1;
                p[q] = rp[at[q]];
            }
            edges(u, p);
        }
        __builtin_amdgcn_wave_barrier();
    }
    return met;
}

// Expansion: every neighbour goes to the output queue.  A tile's edge count
// is its output, so a tile of kDirectEdges and more reserves its place with
// one atomic and writes there in order (the staging areas cost one atomic,
// all on the queue's length, per 2048 edges: 12 k of them, 40 ns each,
// were most of the 25 M-edge expansion of an R-MAT scale 20 search, 545 us
// through staging); smaller tiles go through the waves' staging, which
// gathers many of them per atomic.  Rows of the grid tier reserve theirs when
// they are published.
// A filtering expansion (two-phase levels) runs the filter step that would
// follow on its edges at once: only neighbours whose visited bit is clear go
// to the queue, through the staging, and the edges are counted as the filter
// step's input.  No claims run during an expand step, so the bits are those
// the filter would read.  It saves a grid barrier (a launch) a level and the
// write and read of every edge: two-phase searches of R-MAT scale 19, edge
// factor 24, went from 605 to 489 us, of a 1 M-vertex random tree with
// predecessors from 1150 to 943 us.
constexpr int kDirectEdges = 4096;
// Rows per wave past which the waves of a filtering expansion work alone in a
// persistent loop (two-phase search of R-MAT scale 19, edge factor 24: 449 us
// with workgroup tiles, 389 / 383 / 385 / 385 from 0 / 1 / 4 / 16 rows; scale
// 18, edge factor 8: 282, and 238 / 237 / 240 / 250).  A launch per step has
// two workgroups a CU to cover the tiles' barriers (the 24.4 M-edge step of
// an R-MAT scale 20 hybrid search: 20 us slower with waves alone).
constexpr unsigned kRowsPerWave = 1;

template <bool PRED, bool MAYFILTER = false>
struct Expansion {
    const GraphArgs &g;
    const SearchArgs &s;
    const Cursor c;
    Lds<PRED> &lds;
    WaveQueue<PRED> wq;
    bool direct;  // the current tile's form (workgroup-uniform)
    bool wrote;   // some output did not go through the staging
    bool lost;
    const bool filter, coherent;  // coherent: visited words are read past this XCD's L2
    unsigned long long seen;      // edges met by a filtering expansion (workgroup-uniform)

    __device__ __forceinline__ Expansion(const GraphArgs &g_, const SearchArgs &s_, Cursor c_, Lds<PRED> &lds_,
                                         StepIo io, bool filter_ = false)
        : g(g_), s(s_), c(c_), lds(lds_), wq(make_queue<PRED>(s_, c_.step, lds_, io.light)), direct(false),
          wrote(false), lost(false), filter(MAYFILTER && filter_), coherent(io.stale), seen(0)
    {
    }
    template <int N>
    __device__ __forceinline__ void push_unvisited(const int (&u)[N], const int (&pv)[N])
    {
        unsigned w[N];
#pragma unroll
        for (int j = 0; j < N; j++)
            w[j] = u[j] < 0 ? ~0u : coherent ? ld_agent(s.visited + (u[j] >> 5)) : s.visited[u[j] >> 5];
#pragma unroll
        for (int j = 0; j < N; j++) wq.push(!((w[j] >> (u[j] & 31)) & 1u), u[j], pv[j]);
    }
    // Accounts the filter step's input: its length, and the overflow of an
    // edge queue that could not have held it.
    __device__ __forceinline__ void count_seen()
    {
        if (!filter || threadIdx.x != 0 || seen == 0) return;
        const unsigned long long old = __hip_atomic_fetch_add(&s.ctl->fedges[(c.step + 1) % 3], seen,
                                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(&s.ctl->total_queued, seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old + seen > s.cap) {
            st_agent(wq.overflow, 1u);
            st_agent(wq.overflow_step, 1u);
        }
    }
    __device__ __forceinline__ void put(unsigned at, int u, int par)
    {
        if (at < s.cap) wq.store(at, u, par);
        else lost = true;
    }
    __device__ __forceinline__ void begin(int edges)
    {
        seen += (unsigned long long) edges;
        direct = !filter && edges >= kDirectEdges;
        wrote = wrote || direct;
        // (the row table's barrier orders the word before its readers)
        if (direct && threadIdx.x == 0) lds.ep_base = add_agent(wq.out_len, (unsigned) edges);
    }
    __device__ __forceinline__ void edges(const int (&at)[4], const int (&pv)[4], unsigned x0)
    {
        int u[4];
#pragma unroll
        for (int j = 0; j < 4; j++) u[j] = at[j] >= 0 ? __builtin_nontemporal_load(g.col + at[j]) : -1;
        if (direct) {
            const unsigned base = lds.ep_base + x0;
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (at[j] >= 0) put(base + (unsigned) (j * kBlock), u[j], pv[j]);
        } else if (filter) {
            push_unvisited(u, pv);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) wq.push(at[j] >= 0, u[j], pv[j]);
        }
    }
    template <int K>
    __device__ __forceinline__ void tile(const int (&beg)[K], int (&end)[K], const int (&par)[K], const HubList &hub)
    {
        gather_tile<K>(
            beg, end, par, hub, lds.rt, [&](int e) { begin(e); },
            [&](const int (&at)[4], const int (&pv)[4], unsigned x0) { edges(at, pv, x0); });
    }
    __device__ __forceinline__ HubList hubs(unsigned n, bool enabled) const
    {
        HubList h = hub_list(s, c.step, enabled, n);
        h.out_len = filter ? nullptr : wq.out_len;
        return h;
    }
    __device__ __forceinline__ void hub_chunks()
    {
        hub_phase_chunks<PRED>(s, c, lds, [&](int b, int e, int par) {
            const unsigned out = lds.cta_out;
            int u[kHubChunk / kBlock];
#pragma unroll
            for (int j = 0; j < kHubChunk / kBlock; j++) {
                const int x = b + j * kBlock + (int) threadIdx.x;
                u[j] = x < e ? __builtin_nontemporal_load(g.col + x) : -1;
            }
            if (filter) {
                static_assert(kHubChunk == 4 * kBlock, "a chunk is one round of a workgroup");
                const int pv[4] = {par, par, par, par};
                seen += (unsigned long long) (e - b);
                push_unvisited(u, pv);
                return;
            }
#pragma unroll
            for (int j = 0; j < kHubChunk / kBlock; j++) {
                const int o = j * kBlock + (int) threadIdx.x;
                if (b + o < e) put(out + (unsigned) o, u[j], par);
            }
        });
    }
    __device__ __forceinline__ void report_lost()
    {
        if (lost) {
            st_agent(wq.overflow, 1u);
            st_agent(wq.overflow_step, 1u);
        }
    }
};

template <bool PRED, bool EXACT>
__device__ __forceinline__ void body_contract_expand(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds,
                                     int sub, bool hubs, StepIo io)
{
    Expansion<PRED> x(g, s, c, lds, io);
    bool labeled = false;
    if (sub == 0) {
        const HubList hub = x.hubs(n, hubs);
        // (an item may claim a row of any length: few items go to as many
        // workgroups as runs of the queue allow)
        TileGrab tg = tile_grab(s, n, lds, kItems * kBlock, (n + 15) / 16);
        while (true) {
            const unsigned base = next_tile(&s.ctl->steal[c.step & 1], lds, tg) * tg.width;
            if (base >= n) break;
            int u[kItems], pv[kItems], beg[kItems], end[kItems];
            const unsigned fresh = contract_tile<PRED, EXACT, true>(g, s, c, n, base, tg.width, lds, io, u, pv, beg, end);
            labeled = labeled || fresh != 0;  // (rows of the other items are empty)
            x.template tile<kItems>(beg, end, u, hub);
        }
    } else {
        x.hub_chunks();
    }
    x.report_lost();
    // Vertices labelled here show in the next step's input (prepare_step),
    // unless none of them has neighbours.
    const bool all_staged = !__syncthreads_or(x.wrote);
    finish_step<PRED>(x.wq, lds, s.ctl, c.step, 0u, false, 0, labeled && all_staged, c.iteration);
}

// filter: the filter step runs with it (see Expansion).
template <bool PRED, bool EXACT, bool MAYFILTER = false, bool WAVES = false>
__device__ __forceinline__ void body_expand(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds, int sub,
                            bool hubs, StepIo io, bool filter = false)
{
    Expansion<PRED, MAYFILTER> x(g, s, c, lds, io, filter);
    const int *in = s.q[c.step & 1];
    if (sub == 0 && WAVES && filter && hubs && n > gridDim.x * kWaves * kRowsPerWave) {
        HubList hub = x.hubs(n, hubs);
        if (hub.grid_t != 0x7fffffff) hub.grid_t = min(hub.grid_t, kWaveHubRow);
        const unsigned long long met = wave_rows(
            g, in, n, hub, lds.rt, [&](const auto &u, const auto &p) { x.push_unvisited(u, p); });
        // (fewer than 2^31 edges in all)
        const int sum = wave_inclusive_sum((int) met);
        if (lane_id() == kWave - 1) lds.ep_fe[threadIdx.x / kWave] = (unsigned long long) (unsigned) sum;
        __syncthreads();
        for (int w = 0; w < kWaves; w++) x.seen += lds.ep_fe[w];
        __syncthreads();  // (finish_step writes them again)
    } else if (sub == 0) {
        const HubList hub = x.hubs(n, hubs);
        TileGrab tg = tile_grab(s, n, lds, kBlock, gridDim.x);
        while (true) {
            const unsigned t = next_tile(&s.ctl->steal[c.step & 1], lds, tg);
            if (t >= tg.tiles) break;
            const unsigned i = tg.dealt(t, threadIdx.x);
            int beg[1] = {0}, end[1] = {0}, par[1] = {-1};
            if (threadIdx.x < tg.width && i < n) {
                par[0] = ld_queue(in + i);
                beg[0] = g.row[par[0]];
                end[0] = g.row[par[0] + 1];
            }
            x.template tile<1>(beg, end, par, hub);
        }
    } else {
        x.hub_chunks();
    }
    x.report_lost();
    x.count_seen();
    finish_step<PRED>(x.wq, lds, s.ctl, c.step, 0u, false);
}

// ---------------------------------------------------------------------------
// Chained compaction (config compaction = 2) of the steps whose output per
// tile is bounded by the tile (contract: claim, filter: bitmask cull).  The
// unit of the chain is a grab (the consecutive tiles one tile-counter atomic
// hands a workgroup).  Pass 1 decides every item of the grab and keeps one
// ballot mask per wave and tile in LDS; wave 0 sums the masks, publishes
// the grab's count in its 64-bit status word (epoch, state, value) and finds
// the grab's offset in the output queue by a decoupled look-back over the
// earlier grabs' words (prim::lookback_prefix) -- a single-pass grid scan in
// place of the reference's per-tile atomicAdd reservation
// (util/scan/cooperative_scan.cuh:309-343) and its multi-kernel scan passes.
// Pass 2 re-reads the kept items (still in cache) and writes them at the
// offset plus their rank, so the output keeps the input order.  Grabs are
// taken in increasing order and publish their count before looking back,
// so a grab waits only for grabs already taken, each at most one pass 1
// away.  The last grab stores the output length.
// ---------------------------------------------------------------------------
constexpr unsigned kChainGrabMax = kWave;  // tiles per grab: one lane each in the count scan
static_assert(kChainGrabMax * kWaves * 2 <= kWaves * kWaveQueueCap, "grab masks fit the staging area");

template <bool PRED, bool EXACT, bool FILTER>
__device__ __forceinline__ void chained_step(const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds, StepIo io)
{
    const int *in = s.q[c.step & 1];
    const int *pin = s.pq[c.step & 1];
    int *out = s.q[(c.step + 1) & 1];
    int *pout = PRED ? s.pq[(c.step + 1) & 1] : nullptr;
    // the wave-queue staging is idle: ballot masks [tile][wave]
    unsigned long long *masks = reinterpret_cast<unsigned long long *>(&lds.wq[0][0]);
    int *tile_off = &lds.rt.excl[0][0];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const unsigned tiles = (n + kBlock - 1) / kBlock;
    // (grabs in increasing order, as the look-back needs: always dynamic)
    const unsigned g = min(tile_grab_size(s, tiles), kChainGrabMax);
    const unsigned grabs = (tiles + g - 1) / g;
    const unsigned epoch = (s.scan_epoch + (unsigned) c.step) & 0x3FFFFFFFu;
    while (true) {
        const unsigned first = next_item(&s.ctl->steal[c.step & 1], lds, g);
        if (first >= tiles) break;
        const unsigned cnt = min(g, tiles - first);
        for (unsigned k = 0; k < cnt; k++) {
            const unsigned i = (first + k) * kBlock + threadIdx.x;
            bool keep = false;
            if (i < n) {
                const int u = ld_queue(in + i);
                if (FILTER) {
                    if (u >= 0) {
                        const unsigned w = io.stale ? ld_agent(s.visited + (u >> 5)) : s.visited[u >> 5];
                        keep = ((w >> (u & 31)) & 1u) == 0;
                    }
                } else {
                    const int p = PRED ? ld_queue(pin + i) : -1;
                    keep = u >= 0 && history_pass<PRED>(lds, u) &&
                           claim<EXACT>(s.visited, s.depth, u, s.coherent_filter || io.stale);
                    if (keep) {
                        s.depth[u] = c.iteration;
                        if (PRED) s.pred[u] = p;
                    }
                }
            }
            const unsigned long long m = ballot(keep);
            if (lane == 0) masks[k * kWaves + wave] = m;
        }
        __syncthreads();
        if (wave == 0) {
            int cnt_l = 0;
            if ((unsigned) lane < cnt)
                for (int w = 0; w < kWaves; w++) cnt_l += __popcll(masks[lane * kWaves + w]);
            const int incl = wave_inclusive_sum(cnt_l);
            if ((unsigned) lane < cnt) tile_off[lane] = incl - cnt_l;
            const unsigned agg = (unsigned) readlane(incl, kWave - 1);
            const unsigned j = first / g;
            unsigned prefix = 0;
            if (j == 0) {
                if (lane == 0) prim::publish(s.tile_status, 0, epoch, prim::kStatePrefix, agg);
            } else {
                if (lane == 0) prim::publish(s.tile_status, j, epoch, prim::kStateAggregate, agg);
                prefix = prim::lookback_prefix(s.tile_status, j, epoch);
                if (lane == 0) prim::publish(s.tile_status, j, epoch, prim::kStatePrefix, prefix + agg);
            }
            if (lane == 0) {
                lds.ep_base = prefix;
                if (j == grabs - 1) st_agent(&s.ctl->qlen[(c.step + 1) % 3], prefix + agg);
            }
        }
        __syncthreads();
        const unsigned prefix = lds.ep_base;
        bool lost = false;
        for (unsigned k = 0; k < cnt; k++) {
            const unsigned long long m = masks[k * kWaves + wave];
            if (!((m >> lane) & 1ull)) continue;
            unsigned rank = (unsigned) tile_off[k] + (unsigned) __popcll(m & ((1ull << lane) - 1ull));
            for (int w = 0; w < wave; w++) rank += (unsigned) __popcll(masks[k * kWaves + w]);
            const unsigned i = (first + k) * kBlock + threadIdx.x;
            const unsigned at = prefix + rank;
            if (at < s.cap) {
                const int u = ld_queue(in + i), p = PRED && FILTER ? ld_queue(pin + i) : -1;
                if (io.light) {
                    st_agent(out + at, u);
                    if (PRED) st_agent(pout + at, p);
                } else {
                    out[at] = u;
                    if (PRED) pout[at] = p;
                }
            } else {
                lost = true;
            }
        }
        if (lost) {
            st_agent(&s.ctl->overflow, 1u);
            st_agent(&s.ctl->ovf[(c.step + 1) % 3], 1u);
        }
        // (next_item's barrier orders these mask reads before the next grab's writes)
    }
}

template <bool PRED, bool EXACT>
__device__ __forceinline__ void body_contract(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds,
                                              StepIo io)
{
    WaveQueue<PRED> wq = make_queue<PRED>(s, c.step, lds, io.light);
    if (s.tile_status) {
        chained_step<PRED, EXACT, false>(s, c, n, lds, io);
    } else {
        TileGrab tg = tile_grab(s, n, lds, kItems * kBlock, (n + kBlock - 1) / kBlock);
        while (true) {
            const unsigned base = next_tile(&s.ctl->steal[c.step & 1], lds, tg) * tg.width;
            if (base >= n) break;
            int u[kItems], pv[kItems], ub[kItems], ud[kItems];
            const unsigned fresh =
                contract_tile<PRED, EXACT, false>(g, s, c, n, base, tg.width, lds, io, u, pv, ub, ud);
#pragma unroll
            for (int k = 0; k < kItems; k++) wq.push((fresh >> k) & 1, u[k], -1);
        }
    }
    finish_step<PRED>(wq, lds, s.ctl, c.step, 0u, false);
}

template <bool PRED, bool EXACT>
__device__ __forceinline__ void body_filter(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds,
                                            StepIo io)
{
    (void) g;
    WaveQueue<PRED> wq = make_queue<PRED>(s, c.step, lds, io.light);
    const int *in = s.q[c.step & 1];
    const int *pin = s.pq[c.step & 1];
    if (s.tile_status) {
        chained_step<PRED, EXACT, true>(s, c, n, lds, io);
    } else {
        TileGrab tg = tile_grab(s, n, lds, kItems * kBlock, (n + kBlock - 1) / kBlock);
        while (true) {
            const unsigned base = next_tile(&s.ctl->steal[c.step & 1], lds, tg) * tg.width;
            if (base >= n) break;
            int u[kItems], p[kItems];
            unsigned w[kItems];
#pragma unroll
            for (int k = 0; k < kItems; k++) {
                const unsigned o = (unsigned) (k * kBlock) + threadIdx.x;
                const bool ok = o < tg.width && base + o < n;
                u[k] = ok ? ld_queue(in + base + o) : -1;
                p[k] = PRED && ok ? ld_queue(pin + base + o) : -1;
            }
            // Bitmask only: the history hash is reserved for claims, because a
            // hit there must mean the vertex has already been claimed or found
            // visited by this workgroup.
#pragma unroll
            for (int k = 0; k < kItems; k++)
                w[k] = u[k] < 0 ? ~0u : io.stale ? ld_agent(s.visited + (u[k] >> 5)) : s.visited[u[k] >> 5];
#pragma unroll
            for (int k = 0; k < kItems; k++) wq.push(u[k] >= 0 && !((w[k] >> (u[k] & 31)) & 1u), u[k], p[k]);
        }
    }
    finish_step<PRED>(wq, lds, s.ctl, c.step, 0u, false);
}

// Whether the expand steps of two-phase levels filter too (chained compaction
// filters in the order of its input, in a step of its own).
__device__ __forceinline__ bool filters(const SearchArgs &s) { return s.tile_status == nullptr; }

__device__ __forceinline__ bool gathers(int phase)
{
    return phase == kPhaseExpandContract || phase == kPhaseContractExpand || phase == kPhaseExpand;
}

template <bool PRED, bool EXACT>
__device__ __forceinline__ void run_body(int phase, const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n,
                                         Lds<PRED> &lds, int sub, bool hubs, unsigned long long fe)
{
    const StepIo io{false, false, true};
    switch (phase) {
    case kPhaseExpandContract: body_expand_contract<PRED>(g, s, c, n, lds, sub, hubs, fe, io); break;
    case kPhaseContractExpand: body_contract_expand<PRED, EXACT>(g, s, c, n, lds, sub, hubs, io); break;
    case kPhaseContract: body_contract<PRED, EXACT>(g, s, c, n, lds, io); break;
    case kPhaseExpand: body_expand<PRED, EXACT, true>(g, s, c, n, lds, sub, hubs, io, filters(s)); break;
    case kPhaseBottomUp: body_bottom_up<PRED>(g, s, c, lds); break;
    default: body_filter<PRED, EXACT>(g, s, c, n, lds, io); break;
    }
}

// The phases a persistent loop can run (the others are not compiled into
// its kernel, which keeps their registers out of its budget).
template <bool PRED, bool EXACT, int LOOP>
__device__ __forceinline__ void loop_body(int phase, const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n,
                                          Lds<PRED> &lds, int sub, bool hubs, unsigned long long fe, StepIo io,
                                          unsigned *next_bits = nullptr, bool from_bitmap = false)
{
    if constexpr (LOOP == kLoopEC) {
        body_expand_contract<PRED>(g, s, c, n, lds, sub, hubs, fe, io);
    } else if constexpr (LOOP == kLoopCE) {
        // (expand: the step that ends a contract-expand fast path)
        if (phase == kPhaseExpand) body_expand<PRED, EXACT>(g, s, c, n, lds, sub, hubs, io);
        else body_contract_expand<PRED, EXACT>(g, s, c, n, lds, sub, hubs, io);
    } else if constexpr (LOOP == kLoopDO) {
        if (phase == kPhaseBottomUp) body_bottom_up<PRED>(g, s, c, lds);
        else body_expand_contract<PRED>(g, s, c, n, lds, sub, hubs, fe, io, next_bits, from_bitmap);
    } else {
        if (phase == kPhaseContract) body_contract<PRED, EXACT>(g, s, c, n, lds, io);
        else if (phase == kPhaseExpand)
            body_expand<PRED, EXACT, true, true>(g, s, c, n, lds, sub, hubs, io, filters(s));
        else body_filter<PRED, EXACT>(g, s, c, n, lds, io);
    }
}

// Two grid-wide passes that turn the vertex queue of step c into the
// frontier bitmap fbm[c.iteration & 1] (zero, then set); a grid barrier or
// kernel boundary must separate them.  A persistent search skips the first:
// its prologue clears both bitmaps and queue_from_bitmap clears them again
// whenever the search turns top-down, so they are clear at every top-down
// level.
__device__ __forceinline__ void frontier_bitmap_pass(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n,
                                                     int pass)
{
    unsigned *bm = s.fbm[c.iteration & 1];
    const unsigned stride = gridDim.x * kBlock;
    if (pass == 0) {
        const unsigned words = ((unsigned) g.nodes + 31) >> 5;
        for (unsigned w = blockIdx.x * kBlock + threadIdx.x; w < words; w += stride) bm[w] = 0u;
    } else {
        const int *in = s.q[c.step & 1];
        for (unsigned i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
            int u = ld_queue(in + i);
            __hip_atomic_fetch_or(&bm[u >> 5], 1u << (u & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ---------------------------------------------------------------------------
// Mark-and-compact form of a large top-down step (expand-contract and the
// top-down levels of direction-optimizing search).  The claims of a big
// level are bound by atomic throughput (about 27 G/s on this part, whatever
// the scope), while plain random byte stores run at about 84 G/s.  Such a
// level therefore only marks its discoveries: every edge to a vertex whose
// visited bit is clear (the bits do not change during the pass) stores 1
// into marks[u] -- duplicates merge, as every writer stores the same byte
// -- and, for predecessors, the edge's source into pred[u] (any writer
// leaves a valid parent).  After a grid barrier one streaming pass turns
// the marks of each 32-vertex word into visited bits, labels and queue
// entries (in vertex order) and clears them.  The pass and its barrier cost
// about 10-15 us, so small levels keep the atomic claims.
// ---------------------------------------------------------------------------
constexpr unsigned long long kMarkEdges = 1ull << 20;  // fewest frontier edges for the marked form

__device__ __forceinline__ bool marked_step(const SearchArgs &s, unsigned long long fe)
{
    return s.marks != nullptr && fe >= kMarkEdges && fe >= (unsigned long long) s.nodes / 2;
}

template <bool PRED>
__device__ __forceinline__ void body_expand_mark(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, Lds<PRED> &lds,
                                 int sub, bool hubs)
{
    // An edge marks its target when the target's visited bit is clear.
    const int *in = s.q[c.step & 1];
    if (sub == 0) {
        // Tiles of kBlock frontier vertices: rows of the grid tier are
        // published, the rest of the tile's edges are spread evenly over the
        // workgroup through an LDS degree scan (as in the LDS fast path),
        // four consecutive edges per thread per round with every load of a
        // round in flight -- instead of the gather tiers' one chain per
        // round of 64 edges.
        const HubList hub = hub_list(s, c.step, hubs, n);
        int *tbeg = lds.wq[0];  // the wave-queue staging is idle in a marked step
        int *tpar = lds.wq[1];
        int *toff = lds.wq[2];
        static_assert(kWaveQueueCap >= kBlock && kWaves >= 3, "tile tables fit the staging area");
        TileGrab tg = tile_grab(s, n, lds, kBlock, gridDim.x);
        while (true) {
            const unsigned t = next_tile(&s.ctl->steal[c.step & 1], lds, tg);
            if (t >= tg.tiles) break;
            const unsigned i = tg.dealt(t, threadIdx.x);
            int v = -1, beg = 0, end = 0;
            if (threadIdx.x < tg.width && i < n) {
                v = ld_queue(in + i);
                beg = g.row[v];
                end = g.row[v + 1];
            }
            if (publish_hub_row(beg, end, v, hub)) end = beg;
            int total = 0;
            const int off = block_exclusive_sum(end - beg, lds.ep_scan, &total);
            // (the scan's barriers order the previous tile's reads before these writes)
            tbeg[threadIdx.x] = beg;
            tpar[threadIdx.x] = v;
            toff[threadIdx.x] = off;
            __syncthreads();
            for (int b0 = 0; b0 < total; b0 += kBlock * 4) {
                const int e0 = b0 + (int) threadIdx.x * 4;
                int r = 0;
                if (e0 < total) {  // last row with off <= e0 (it has edges)
                    int lo = 0, hi = kBlock - 1;
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (toff[mid] <= e0) lo = mid;
                        else hi = mid - 1;
                    }
                    r = lo;
                }
                int at[4], pv[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int e = e0 + j;
                    at[j] = -1;
                    pv[j] = -1;
                    if (e < total) {
                        while (r + 1 < kBlock && toff[r + 1] <= e) r++;
                        at[j] = tbeg[r] + (e - toff[r]);
                        pv[j] = tpar[r];
                    }
                }
                int u[4];
                unsigned w[4];
#pragma unroll
                for (int j = 0; j < 4; j++) u[j] = at[j] >= 0 ? g.col[at[j]] : -1;
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = u[j] >= 0 ? s.visited[u[j] >> 5] : ~0u;
                bool todo[4];
#pragma unroll
                for (int j = 0; j < 4; j++) todo[j] = u[j] >= 0 && !((w[j] >> (u[j] & 31)) & 1u);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (todo[j]) {
                        s.marks[u[j]] = 1;
                        if (PRED) s.pred[u[j]] = pv[j];
                    }
                }
            }
        }
        return;
    }
    // Grid-tier chunks, four workgroup-widths of edges per round with every
    // load of a round in flight together (the per-edge chain -- column,
    // visited word, mark -- is the cost of these levels, not bytes).
    constexpr int U = 4;
    hub_phase_chunks<PRED>(s, c, lds, [&](int b, int e, int pv) {
        for (int k = b; k < e; k += U * kBlock) {
            int u[U];
            unsigned w[U];
#pragma unroll
            for (int j = 0; j < U; j++) {
                const int idx = k + j * kBlock + (int) threadIdx.x;
                u[j] = idx < e ? g.col[idx] : -1;
            }
#pragma unroll
            for (int j = 0; j < U; j++) w[j] = u[j] >= 0 ? s.visited[u[j] >> 5] : ~0u;
            bool todo[U];
#pragma unroll
            for (int j = 0; j < U; j++) todo[j] = u[j] >= 0 && !((w[j] >> (u[j] & 31)) & 1u);
#pragma unroll
            for (int j = 0; j < U; j++) {
                if (todo[j]) {
                    s.marks[u[j]] = 1;
                    if (PRED) s.pred[u[j]] = pv;
                }
            }
        }
    });
}

// Bits of the four 0/1 bytes of x.
__device__ __forceinline__ unsigned byte_bits(unsigned x)
{
    return (x & 1u) | ((x >> 7) & 2u) | ((x >> 14) & 4u) | ((x >> 21) & 8u);
}

// Grid-wide; follows the marking pass behind a grid barrier, and a grid
// barrier must follow it.  Appends to the queue of step c + 1 like the
// claiming form (one reservation per workgroup and word batch), in vertex
// order.  With fbm_out set, also writes every word of that frontier bitmap
// (the next step's frontier, exactly: a direction-optimizing search that
// turns bottom-up next needs no bitmap pass).
template <bool PRED>
__device__ __forceinline__ void mark_compact(const GraphArgs &g, const SearchArgs &s, Cursor c, Lds<PRED> &lds, unsigned *fbm_out)
{
    const unsigned words = ((unsigned) g.nodes + 31) >> 5;
    const int next_depth = c.iteration + 1;
    int *out = s.q[(c.step + 1) & 1];
    // the new vertices of a word batch, staged in the (idle) wave-queue LDS
    int *stage = &lds.wq[0][0];
    constexpr int kStage = kWaves * kWaveQueueCap;
    unsigned fe = 0;
    bool over = false;
    for (unsigned w0 = blockIdx.x * kBlock; w0 < words; w0 += gridDim.x * kBlock) {
        const unsigned w = w0 + threadIdx.x;
        unsigned bits = 0;
        if (w < words) {
            uint4 *m = reinterpret_cast<uint4 *>(s.marks + 32ull * w);
            const uint4 lo = m[0], hi = m[1];
            bits = byte_bits(lo.x) | byte_bits(lo.y) << 4 | byte_bits(lo.z) << 8 | byte_bits(lo.w) << 12 |
                   byte_bits(hi.x) << 16 | byte_bits(hi.y) << 20 | byte_bits(hi.z) << 24 | byte_bits(hi.w) << 28;
            if (bits) {
                m[0] = make_uint4(0u, 0u, 0u, 0u);
                m[1] = make_uint4(0u, 0u, 0u, 0u);
                const unsigned vis = s.visited[w];
                bits &= ~vis;
                if (bits) s.visited[w] = vis | bits;
            }
            if (fbm_out) fbm_out[w] = bits;
        }
        int total = 0;
        const int excl = block_exclusive_sum(__popc(bits), lds.ep_scan, &total);
        if (total == 0) continue;  // block-uniform
        if (threadIdx.x == 0) lds.ep_base = add_agent(&s.ctl->qlen[(c.step + 1) % 3], (unsigned) total);
        if (total <= kStage) {
            // labels, queue entries and degrees spread over the workgroup,
            // four vertices per thread per round with their row loads in
            // flight together (a thread's own word may hold 32)
            int k = excl;
            for (unsigned b = bits; b; b &= b - 1) stage[k++] = (int) ((w << 5) + (unsigned) __builtin_ctz(b));
            __syncthreads();
            const unsigned base = lds.ep_base;
            for (int i0 = 4 * (int) threadIdx.x; i0 < total; i0 += 4 * kBlock) {
                int v[4], r0[4], r1[4];
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = i0 + j < total ? stage[i0 + j] : -1;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    r0[j] = v[j] >= 0 && s.track_edges ? g.row[v[j]] : 0;
                    r1[j] = v[j] >= 0 && s.track_edges ? g.row[v[j] + 1] : 0;
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (v[j] < 0) continue;
                    s.depth[v[j]] = next_depth;
                    const unsigned pos = base + (unsigned) (i0 + j);
                    if (pos < s.cap) out[pos] = v[j];
                    else over = true;
                    fe += (unsigned) (r1[j] - r0[j]);
                }
            }
        } else {
            __syncthreads();
            unsigned pos = lds.ep_base + (unsigned) excl;
            for (unsigned b = bits; b; b &= b - 1) {
                const int v = (int) ((w << 5) + (unsigned) __builtin_ctz(b));
                s.depth[v] = next_depth;
                if (s.track_edges) fe += (unsigned) (g.row[v + 1] - g.row[v]);
                if (pos < s.cap) out[pos] = v;
                else over = true;
                pos++;
            }
        }
        __syncthreads();  // ep_base and the stage are reused by the next batch
    }
    if (over) {
        st_agent(&s.ctl->overflow, 1u);
        st_agent(&s.ctl->ovf[(c.step + 1) % 3], 1u);
    }
    // frontier-edge counter: one update per workgroup
    WaveQueue<PRED> wq = make_queue<PRED>(s, c.step, lds);
    finish_step<PRED>(wq, lds, s.ctl, c.step, fe, s.track_edges != 0);
}

// Direction choice of a direction-optimizing search at the top of a level
// (grid-uniform: every input is read after the level barrier).
//
// ve is the caller's running sum of fedges over the steps up to this one.
// The global visited_edges total must not be read here: workgroups already
// in this level's body keep adding to it, and a workgroup reading it late
// could choose the other direction -- and then a different sequence of grid
// barriers than the rest of the grid.
// Direction rule: mf = the frontier's edges, n = its vertices, ve = edges
// visited so far, prev_mf = the previous frontier's edges.  A top-down
// search turns bottom-up only while its frontier grows (Beamer et al.'s
// growing phase): near the end of a high-diameter search the unexplored
// edges fall below alpha times a shrinking frontier's, and a bottom-up
// level there would turn straight back.
__device__ __forceinline__ int direction_rule(const SearchArgs &s, int phase, unsigned long long mf, unsigned n,
                                              unsigned long long ve, unsigned long long prev_mf)
{
    unsigned long long mu = s.total_edges > ve ? s.total_edges - ve : 0ull;
    if (phase == kPhaseExpandContract) {
        if (mf > prev_mf && mf * (unsigned long long) s.do_alpha > mu) return kPhaseBottomUp;
    } else if ((unsigned long long) n * (unsigned long long) s.do_beta < (unsigned long long) s.nodes) {
        return kPhaseExpandContract;
    }
    return phase;
}


// Whether a level is small enough for the single-workgroup fast path.
// fe: the step's frontier edges (used when they are tracked).
__device__ __forceinline__ bool fast_level(const SearchArgs &s, Cursor c, unsigned n, unsigned long long fe)
{
    if (s.fast_t < 0 || n > (unsigned) s.fast_t || c.phase == kPhaseBottomUp) return false;
    if (s.track_edges && fe > 32ull * (unsigned) s.fast_t) return false;
    return true;
}

__device__ __forceinline__ bool fast_level(const SearchArgs &s, Cursor c, unsigned n)
{
    return fast_level(s, c, n, s.track_edges ? ld64_agent(&s.ctl->fedges[c.step % 3]) : 0ull);
}

// filtered: a two-phase expand step ran the filter as well.
__device__ __forceinline__ Cursor advance(int loop, Cursor c, bool filtered = false)
{
    c.step++;
    if (loop != kLoopTP) {
        // (a contract-expand loop returns to contract-expand after the
        // expand step that ends its fast path: the expanded members were
        // labelled with c.iteration, their neighbours get c.iteration + 1)
        c.iteration++;
        if (loop == kLoopCE) c.phase = kPhaseContractExpand;
    } else {
        if (c.phase == kPhaseContract) c.phase = kPhaseExpand;
        else if (c.phase == kPhaseExpand && !filtered) c.phase = kPhaseFilter;
        else { c.phase = kPhaseContract; c.iteration++; }
    }
    return c;
}

// Counter maintenance for step c (one thread): zero the counters the next
// step appends to / steals from, and account the input length.
__device__ __forceinline__ void prepare_step(Control *ctl, Cursor c, unsigned n)
{
    st_agent(&ctl->qlen[(c.step + 2) % 3], 0u);
    st_agent(&ctl->steal[(c.step + 1) & 1], 0u);
    st_agent(&ctl->hub_steal[(c.step + 1) & 1], 0u);
    st_agent(&ctl->compact, 0u);
    st_agent(&ctl->ovf[(c.step + 2) % 3], 0u);
    __hip_atomic_store(&ctl->hub_alloc[(c.step + 1) & 1], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ctl->fedges[(c.step + 2) % 3], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(&ctl->total_queued, (unsigned long long) n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // deepest label so far: the members of a vertex frontier carry the step's
    // iteration, those whose neighbours form an edge frontier the one before
    const bool members = c.phase == kPhaseExpandContract || c.phase == kPhaseBottomUp || c.phase == kPhaseExpand;
    if (n > 0) atomicMax(&ctl->max_depth, members ? c.iteration : c.iteration - 1);
    if (c.step < kLevelLog) {
        ctl->level_len[c.step] = n;
        ctl->level_clock[c.step] = wall_clock64();
    }
}

__device__ __forceinline__ unsigned frontier_length(const SearchArgs &s, int step)
{
    unsigned n = ld_agent(&s.ctl->qlen[step % 3]);
    return n < s.cap ? n : s.cap;
}

__device__ __forceinline__ bool hubs_pending(const SearchArgs &s, int step)
{
    return __hip_atomic_load(&s.ctl->hub_alloc[step & 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0ull;
}

// ---------------------------------------------------------------------------
// LDS-resident fast path of the vertex-frontier loops (expand-contract and
// the top-down levels of direction-optimizing search).  Block 0 alone runs
// consecutive small levels while the rest of the grid waits at a grid
// barrier.  The frontier, its members' row starts and degrees stay in LDS
// between levels, and the global queue and counters are written once, when
// the path ends.  The level's edges are spread evenly over the threads, each
// taking kFastK consecutive edges through the exclusive degree scan, and each
// memory trip of a batch is issued for all kFastK edges before the first
// result is used: column index, visited word, claim, row bounds -- four
// dependent trips per batch, and a level of up to kBlock * kFastK edges is
// one batch.  A high-diameter graph spends its whole search here.
// ---------------------------------------------------------------------------
constexpr int kFastCap = 1024;  // frontier members kept in LDS
constexpr int kFastK = 4;       // consecutive edges per thread per batch
// Most edges of a level run by the path: a batch of kBlock * kFastK edges
// costs about one quarter of a grid-wide step, so a few batches still win.
constexpr unsigned long long kFastEdges = 4ull * kBlock * kFastK;
static_assert(kFastCap <= 4 * kBlock, "the degree scan takes four members per thread");

// Direct levels: when every member's degree is small, groups of lanes take
// whole rows (a thread up to kFastDirect edges) with no degree scan and no
// search for each edge's member.
constexpr int kFastDirect = 8;
static_assert(kFastDirect == 8, "fast_direct_lg spans one to eight lanes per member");

// log2 of the lanes per member of a direct level whose members' largest
// degree is maxd (30: too large for one)
__device__ __forceinline__ int fast_direct_lg(int maxd)
{
    return maxd <= 1 ? 0 : maxd <= 2 ? 1 : maxd <= 4 ? 2 : maxd <= kFastDirect ? 3 : 30;
}

__device__ __forceinline__ bool fast_direct(int maxd, unsigned n)
{
    const int lg = fast_direct_lg(maxd);
    return lg < 30 && ((int) n << lg) <= kBlock * kFastDirect;
}

struct FastFront {
    int v[2][kFastCap];
    int beg[2][kFastCap];
    int deg[2][kFastCap];        // degree on append; the level's exclusive scan in place
    int maxdeg[2];               // largest degree of each buffer's members
    unsigned count;              // next-frontier appends
    unsigned dups;               // two-phase: further edges to vertices claimed in the level
    unsigned long long fe;       // next frontier's edges
    int labeled;
    int scan[kWaves];            // per-wave sums of the degree scan
    unsigned long long wfe[kWaves];
    int wlab[kWaves];
    int wmax[kWaves];
};

// FASTV: the fast path's copy of the visited bitmap takes the rest of the
// workgroup's LDS (gfx950: 160 KiB) once the frontier buffers and 1 KiB for
// the level loop's other variables are placed: graphs of up to
// kFastVisitedWords * 32 vertices.  Larger graphs launch the instantiation
// without it, which keeps the smaller LDS footprint.
constexpr int kLdsBytes = 163840;
constexpr int kFastVisitedWords = ((kLdsBytes - 1024 - (int) sizeof(FastFront)) / 4) & ~63;
static_assert(kFastVisitedWords * 32 == BFS_FAST_VISITED_MAX, "the header states the fast path's LDS bitmap size");

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <bool FASTV>
struct FastLds {
    FastFront f;
    __attribute__((aligned(16))) unsigned vbits[FASTV ? kFastVisitedWords : 4];
};

// The level loop's LDS: the step bodies' staging and the fast path's
// frontier are never live at once (the fast path starts after a grid
// barrier and re-initialises the step state when it ends).
template <bool PRED, bool FASTV>
union LoopLds {
    Lds<PRED> step;
    FastLds<FASTV> fast;
};

// Exclusive scan of F.deg[b][0, n) in place; returns the sum to every thread.
__device__ int fast_scan(FastFront &F, int b, unsigned n)
{
    const unsigned t0 = 4u * threadIdx.x;
    int d[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        d[k] = t0 + k < n ? F.deg[b][t0 + k] : 0;
        sum += d[k];
    }
    int total;
    int off = block_exclusive_sum(sum, F.scan, &total);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (t0 + k < n) F.deg[b][t0 + k] = off;
        off += d[k];
    }
    __syncthreads();
    return total;
}

// kFastK consecutive edges from e0 (one thread's share of a batch) of an
// LDS-resident frontier: offs = the exclusive scan of its n members' degrees
// (total edges in all), begs = their row starts, vs = the members.  Returns
// fast_claim_slots' mask; pv[k] = the owner of slot k's row.
template <bool PRED, bool EXACT, bool LOCAL>
__device__ __forceinline__ unsigned fast_edges(const GraphArgs &g, const SearchArgs &s, int next_depth,
                                               const int *offs, const int *begs, const int *vs, unsigned n,
                                               int total, int e0, int (&u)[kFastK], int (&pv)[kFastK],
                                               int (&ub)[kFastK], int (&ud)[kFastK], bool ldsv = false,
                                               unsigned *vbits = nullptr, StepIo io = StepIo{false, false})
{
    // member holding edge e0: the last i with offs[i] <= e0 (it has edges)
    int i = 0;
    if (e0 < total) {
        int lo = 0, hi = (int) n - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (offs[mid] <= e0) lo = mid;
            else hi = mid - 1;
        }
        i = lo;
    }
    // column positions first (LDS only): a loop between two global
    // loads makes the compiler wait for the first
    int at[kFastK];
#pragma unroll
    for (int k = 0; k < kFastK; k++) {
        const int e = e0 + k;
        at[k] = -1;
        pv[k] = -1;
        if (e < total) {
            while (i + 1 < (int) n && offs[i + 1] <= e) i++;
            at[k] = begs[i] + (e - offs[i]);
            pv[k] = vs[i];
        }
    }
    return fast_claim_slots<PRED, EXACT, LOCAL, kFastK>(g, s, next_depth, at, pv, u, ub, ud, ldsv, vbits, io);
}

// Appends one thread's claimed slots to LDS buffer dst (one LDS reservation
// per wave); members past kFastCap go to the global queue `spill` at the
// same positions.  Wave-converged.
template <int S>
__device__ __forceinline__ void fast_append(const SearchArgs &s, FastFront &F, int dst, int *spill, unsigned fresh,
                                            const int (&u)[S], const int (&ub)[S], const int (&ud)[S],
                                            unsigned long long &fe, bool &labeled, int &dmax)
{
    const int cnt = __popc(fresh);
    const int incl = wave_inclusive_sum(cnt);
    const int wtot = readlane(incl, kWave - 1);
    if (!wtot) return;
    unsigned base = 0;
    if (lane_id() == 0) base = atomicAdd(&F.count, (unsigned) wtot);
    unsigned p = (unsigned) readlane((int) base, 0) + (unsigned) (incl - cnt);
#pragma unroll
    for (int k = 0; k < S; k++) {
        if ((fresh >> k) & 1) {
            const int d = ud[k] - ub[k];
            fe += (unsigned) d;
            dmax = max(dmax, d);
            labeled = true;
            if (p < (unsigned) kFastCap) {
                F.v[dst][p] = u[k];
                F.beg[dst][p] = ub[k];
                F.deg[dst][p] = d;
            } else if (p < s.cap) {
                spill[p] = u[k];
            }
            p++;
        }
    }
}

// Folds the threads' edge sums, label flags and largest degrees of the
// members just appended to buffer dst into F.fe, F.labeled, F.maxdeg[dst].
// Every thread calls it.
__device__ __forceinline__ void fast_fold(FastFront &F, int dst, unsigned long long fe, bool labeled, int dmax)
{
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int lo = wave_inclusive_sum((int) (fe & 0xFFFFu));
    const int hi = wave_inclusive_sum((int) (fe >> 16));
    const int wmax = wave_inclusive_max_nonneg(dmax);
    const bool any = ballot(labeled) != 0;
    if (lane == kWave - 1) {
        F.wfe[wave] = ((unsigned long long) (unsigned) hi << 16) + (unsigned long long) (unsigned) lo;
        F.wlab[wave] = any ? 1 : 0;
        F.wmax[wave] = wmax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long f = 0;
        int l = 0, dm = 0;
        for (int w = 0; w < kWaves; w++) {
            f += F.wfe[w];
            l |= F.wlab[w];
            dm = max(dm, F.wmax[w]);
        }
        F.fe = f;
        F.labeled = l;
        F.maxdeg[dst] = dm;
    }
    __syncthreads();
}

// One level from LDS buffer src (n members, 0 < n <= kFastCap) into buffer
// src ^ 1; members past kFastCap go to the global queue `spill` (the one the
// step after the path reads) at the same positions.  When the members' rows fit kFastDirect slots per thread
// (every lattice level), each member's row goes to a group of consecutive
// lanes, one edge per lane; otherwise the level's edges are spread evenly
// over the threads through the degree scan, kFastK per thread per batch.
// Every thread calls it.
// count_dups (direct levels only): also counts in F.dups the edges, other
// than the claiming ones, whose targets the level claimed.
template <bool PRED, bool EXACT>
__device__ __forceinline__ void fast_lds_level(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, int src,
                                               FastFront &F, bool ldsv, unsigned *vbits, int *spill,
                                               bool count_dups = false)
{
    const int dst = src ^ 1;
    const int next_depth = c.iteration + 1;
    const int maxd = F.maxdeg[src];
    if (threadIdx.x == 0) {
        F.count = 0;
        F.dups = 0;
    }
    unsigned long long fe = 0;
    bool labeled = false;
    int dmax = 0;
    // Direct level: 2^lg consecutive lanes per member (2^lg >= its largest
    // degree), lane k of a group taking edge k, so that the column entries
    // one load instruction reads are whole rows side by side; kFastDirect
    // such passes cover up to kBlock * kFastDirect / 2^lg members.
    const int lg = fast_direct_lg(maxd);
    if (fast_direct(maxd, n)) {
        __syncthreads();  // the resets above precede every append
        int at[kFastDirect], pv[kFastDirect];
        const int k = (int) threadIdx.x & ((1 << lg) - 1);
        const int i0 = (int) threadIdx.x >> lg;
#pragma unroll
        for (int j = 0; j < kFastDirect; j++) {
            const int i = i0 + ((j * kBlock) >> lg);
            at[j] = -1;
            pv[j] = -1;
            if (i < (int) n && k < F.deg[src][i]) {
                at[j] = F.beg[src][i] + k;
                pv[j] = F.v[src][i];
            }
        }
        int u[kFastDirect], ub[kFastDirect], ud[kFastDirect];
        const unsigned fresh =
            fast_claim_slots<PRED, EXACT, true, kFastDirect>(g, s, next_depth, at, pv, u, ub, ud, ldsv, vbits);
        fast_append<kFastDirect>(s, F, dst, spill, fresh, u, ub, ud, fe, labeled, dmax);
        if (count_dups) {
            fast_fold(F, dst, fe, labeled, dmax);
            // (after the fold's barriers every label of the level is
            // visible to the workgroup)
            int dep[kFastDirect];
#pragma unroll
            for (int j = 0; j < kFastDirect; j++)
                dep[j] = u[j] >= 0 && !((fresh >> j) & 1) ? s.depth[u[j]] : -1;
            int d = 0;
#pragma unroll
            for (int j = 0; j < kFastDirect; j++) d += dep[j] == next_depth ? 1 : 0;
            const int wsum = wave_inclusive_sum(d);
            if (lane_id() == kWave - 1 && wsum) atomicAdd(&F.dups, (unsigned) wsum);
            __syncthreads();
            return;
        }
    } else {
        const int total = fast_scan(F, src, n);  // (its barriers order the resets before the appends)
        for (int b0 = 0; b0 < total; b0 += kBlock * kFastK) {
            int u[kFastK], pv[kFastK], ub[kFastK], ud[kFastK];
            const unsigned fresh =
                fast_edges<PRED, EXACT, true>(g, s, next_depth, F.deg[src], F.beg[src], F.v[src], n, total,
                                              b0 + (int) threadIdx.x * kFastK, u, pv, ub, ud, ldsv, vbits);
            fast_append<kFastK>(s, F, dst, spill, fresh, u, ub, ud, fe, labeled, dmax);
        }
    }
    fast_fold(F, dst, fe, labeled, dmax);
}

// ---------------------------------------------------------------------------
// Bit marks: the large top-down and contraction steps of graphs whose
// visited bitmap fits the workgroup's LDS (FASTV).  A workgroup sets the bits
// of the targets of its share of the step's edges (or queue items) in an LDS
// bitmap of all vertices, writes the bitmap to its slab in device memory, and
// after a grid barrier every workgroup ORs its range of words over all the
// slabs: new vertices are the bits not visited yet, and get their labels,
// queue entries (in vertex order) and degree sums there, as in mark_compact.
//
// An LDS atomic costs a few cycles where a claim costs the device 1/27 ns and
// a byte mark 1/84 ns, so the marking streams the columns; the price is the
// slabs, V / 8 bytes per workgroup written and read once (64 MB at 2^20
// vertices), past the L2 so that a light barrier orders them.
// R-MAT scale 20, edge factor 16 (31 M edges): expand-contract 430 -> 313 us,
// its 24.9 M-edge level 190 -> 135 us; a contraction of 5.1 M queued edges
// 133 -> 25 us (hybrid 800 -> 650 us, contract-expand 1140 -> 600 us).
// ---------------------------------------------------------------------------
struct BitLds {
    RowTable rt;
    int list[64 * kWave];            // new vertices of 128 words
    unsigned acc[2 * kWave];         // the words being collected
    unsigned base;
    int scan[kWaves];
    unsigned long long wfe[kWaves];
};
static_assert(sizeof(BitLds) <= sizeof(FastFront), "the bitmap stays free of the step's other variables");

// Whether a step of `work` edges or items takes bit marks (grid-uniform).  The
// passes over the slabs cost 10 us and more with V (30 us at 2^20 vertices);
// claims cost the more the fewer lines the bitmap has, as atomics on a line
// serialise (69 k claims of a 100 k-vertex graph take 18 us, as many as 27
// G/s would do in 2.5).
__device__ __forceinline__ bool bit_step(const SearchArgs &s, unsigned long long work)
{
    return s.slabs != nullptr && gridDim.x <= (unsigned) s.slab_count && s.nodes <= kFastVisitedWords * 32 &&
           work >= bit_mark_work(s.nodes);
}

template <bool PRED, bool EXACT>
__device__ __forceinline__ void bit_mark(const SearchArgs &s, unsigned *vbits, int u, int par)
{
    const unsigned bit = 1u << (u & 31);
    if (PRED) {
        // the workgroup's first edge to an unvisited vertex leaves its source
        // (any of the level's sources is a valid parent)
        const unsigned old =
            __hip_atomic_fetch_or(vbits + (u >> 5), bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (!(old & bit) && !((s.visited[u >> 5] >> (u & 31)) & 1u) && (EXACT || s.depth[u] == -1)) s.pred[u] = par;
    } else {
        __hip_atomic_fetch_or(vbits + (u >> 5), bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

__device__ __forceinline__ void bits_clear(const SearchArgs &s, unsigned *vbits)
{
    const int chunks = (s.nodes + 127) >> 7;
    uint4 *p = reinterpret_cast<uint4 *>(vbits);
    for (int i = threadIdx.x; i < chunks; i += kBlock) p[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
}
static_assert(kFastVisitedWords % 4 == 0, "the bitmap is cleared 16 bytes at a time");

// Marks the targets of the rows of the vertex frontier of step c (the rows
// published for the grid tier follow in bits_from_hubs, behind a barrier).
template <bool PRED>
__device__ __forceinline__ void bits_from_rows(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n,
                                               BitLds &B, unsigned *vbits)
{
    HubList hub = hub_list(s, c.step, true, n);
    hub.grid_t = min(s.grid_t, kWaveHubRow);
    wave_rows(g, s.q[c.step & 1], n, hub, B.rt, [&](const auto &u, const auto &p) {
#pragma unroll
        for (int q = 0; q < (int) (sizeof(u) / sizeof(u[0])); q++)
            if (u[q] >= 0) bit_mark<PRED, true>(s, vbits, u[q], p[q]);
    });
}

// Index of the last grid-tier entry whose first chunk is <= ch, by the whole
// wave: 64 probes at a time, so even a full list takes three dependent loads.
__device__ __forceinline__ unsigned hub_entry_of_wave(const HubEntry *list, unsigned entries, unsigned ch)
{
    unsigned lo = 0, count = entries;
    while (count > 1) {
        const unsigned step = (count + kWave - 1) / kWave;
        const unsigned at = (unsigned) lane_id() * step;
        const uint64_t below = ballot(at < count && list[lo + at].first_chunk <= ch);
        const unsigned k = (unsigned) __popcll(below) - 1u;  // (probe 0 is always below)
        lo += k * step;
        count = min(step, count - k * step);
    }
    return lo;
}

// The published rows, a wave per chunk.
template <bool PRED>
__device__ __forceinline__ void bits_from_hubs(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned *vbits)
{
    const unsigned long long a = ld64_agent(&s.ctl->hub_alloc[c.step & 1]);
    const unsigned entries = min((unsigned) (a >> 32), s.hub_cap);
    if (entries == 0) return;
    const HubEntry *list = s.hubs[c.step & 1];
    const HubEntry last = list[entries - 1];
    const unsigned total = last.first_chunk + (unsigned) ((last.end - last.beg + kHubChunk - 1) / kHubChunk);
    for (unsigned ch = (threadIdx.x / kWave) * gridDim.x + blockIdx.x; ch < total; ch += gridDim.x * kWaves) {
        const HubEntry e = list[hub_entry_of_wave(list, entries, (unsigned) uniform((int) ch))];
        const int b = e.beg + (int) (ch - e.first_chunk) * kHubChunk;
        const int end = min(e.end, b + kHubChunk);
        constexpr int U = 8;
        for (int k = b; k < end; k += U * kWave) {
            int u[U];
#pragma unroll
            for (int j = 0; j < U; j++) {
                const int x = k + j * kWave + lane_id();
                u[j] = x < end ? __builtin_nontemporal_load(g.col + x) : -1;
            }
#pragma unroll
            for (int j = 0; j < U; j++)
                if (u[j] >= 0) bit_mark<PRED, true>(s, vbits, u[j], e.par);
        }
    }
}

// Marks the items of the edge frontier of step c (with their parents).
template <bool PRED, bool EXACT>
__device__ __forceinline__ void bits_from_items(const SearchArgs &s, Cursor c, unsigned n, unsigned *vbits)
{
    const int *in = s.q[c.step & 1];
    const int *pin = s.pq[c.step & 1];
    constexpr unsigned U = 8;
    for (unsigned long long base = blockIdx.x * (unsigned long long) (U * kBlock); base < n;
         base += gridDim.x * (unsigned long long) (U * kBlock)) {
        int u[U], p[U];
#pragma unroll
        for (unsigned j = 0; j < U; j++) {
            const unsigned long long i = base + j * kBlock + threadIdx.x;
            u[j] = i < n ? ld_queue(in + i) : -1;
            p[j] = PRED && i < n ? ld_queue(pin + i) : -1;
        }
#pragma unroll
        for (unsigned j = 0; j < U; j++)
            if (u[j] >= 0) bit_mark<PRED, EXACT>(s, vbits, u[j], p[j]);
    }
}

// Writes the bitmap to the workgroup's slab (a light barrier may follow).
__device__ __forceinline__ void bits_dump(const SearchArgs &s, const unsigned *vbits)
{
    __syncthreads();
    const int pairs = ((s.nodes + 127) >> 7) * 2;
    const unsigned long long *from = reinterpret_cast<const unsigned long long *>(vbits);
    unsigned long long *to =
        reinterpret_cast<unsigned long long *>(s.slabs) + 2 * (size_t) blockIdx.x * slab_quads(s.nodes);
    for (int i = threadIdx.x; i < pairs; i += kBlock)
        __hip_atomic_store(to + i, from[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Collects the slabs behind a grid barrier and a refresh of the caches: new vertices get label `depth`,
// a place in `out` (whose length is *out_len, overflow flags at step + 1)
// and, with fbm_out, their bit in every word of that frontier bitmap; with
// track their degrees are added to fedges.  A full grid barrier must follow,
// or with `through` a light one.
template <bool EXACT>
__device__ __forceinline__ void bits_collect(const GraphArgs &g, const SearchArgs &s, Cursor c, int depth, BitLds &B,
                                             int *out, unsigned *out_len, unsigned *fbm_out, bool track,
                                             bool through = false)
{
    const int words = (s.nodes + 31) >> 5;
    const int quads = (words + 3) >> 2;
    const size_t stride = slab_quads(s.nodes);
    const int per = (quads + (int) gridDim.x - 1) / (int) gridDim.x;
    const int p0 = (int) blockIdx.x * per, p1 = min(quads, p0 + per);
    const int tid = threadIdx.x;
    unsigned fe = 0;
    bool over = false;
    __syncthreads();
    for (int pb = p0; pb < p1; pb += kWave / 2) {
        const int np = min(kWave / 2, p1 - pb);
        if (tid < 2 * kWave) B.acc[tid] = 0u;
        __syncthreads();
        // P lanes (a power of two) cover the quads, the rest of the workgroup
        // further slabs, sixteen loads a thread in flight
        int lg = 0;
        while ((1 << lg) < np) lg++;
        const int lp = tid & ((1 << lg) - 1);
        const int groups = kBlock >> lg;
        if (lp < np) {
            u32x4 a = {0u, 0u, 0u, 0u};
            const u32x4 *from = reinterpret_cast<const u32x4 *>(s.slabs) + pb + lp;
            const int count = (int) gridDim.x;
            for (int sl = tid >> lg; sl < count; sl += 16 * groups) {
                u32x4 v[16];
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    v[j] = u32x4{0u, 0u, 0u, 0u};
                    if (sl + j * groups < count)
                        v[j] = __builtin_nontemporal_load(from + (size_t) (sl + j * groups) * stride);
                }
#pragma unroll
                for (int j = 0; j < 16; j++) a |= v[j];
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (a[j]) atomicOr(&B.acc[4 * lp + j], a[j]);
        }
        __syncthreads();
        const int w = 4 * pb + tid;
        unsigned bits = 0;
        if (tid < 4 * np && w < words) {
            bits = B.acc[tid];
            const unsigned vis = s.visited[w];
            bits &= ~vis;
            if (!EXACT) {
                // chained contractions may have lost bits of labelled vertices
                for (unsigned b = bits; b; b &= b - 1) {
                    const int v = (w << 5) + __builtin_ctz(b);
                    if (s.depth[v] != -1) bits &= ~(1u << (v & 31));
                }
            }
            if (through) {
                if (bits) st_agent(s.visited + w, vis | bits);
                if (fbm_out) st_agent(fbm_out + w, bits);
            } else {
                if (bits) s.visited[w] = vis | bits;
                if (fbm_out) fbm_out[w] = bits;
            }
        }
        int total = 0;
        int k = block_exclusive_sum(__popc(bits), B.scan, &total);
        if (total == 0) continue;  // workgroup-uniform
        if (tid == 0) B.base = add_agent(out_len, (unsigned) total);
        for (unsigned b = bits; b; b &= b - 1) B.list[k++] = (w << 5) + __builtin_ctz(b);
        __syncthreads();
        const unsigned base = B.base;
        for (int i0 = 0; i0 < total; i0 += 4 * kBlock) {
            int v[4], r0[4], r1[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = i0 + j * kBlock + tid;
                v[j] = i < total ? B.list[i] : -1;
                r0[j] = v[j] >= 0 && track ? g.row[v[j]] : 0;
                r1[j] = v[j] >= 0 && track ? g.row[v[j] + 1] : 0;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (v[j] < 0) continue;
                s.depth[v[j]] = depth;
                const unsigned pos = base + (unsigned) (i0 + j * kBlock + tid);
                if (pos >= s.cap) over = true;
                else if (through) st_agent(out + pos, v[j]);
                else out[pos] = v[j];
                fe += (unsigned) (r1[j] - r0[j]);
            }
        }
        __syncthreads();  // the list and the words are used again
    }
    if (over) {
        st_agent(&s.ctl->overflow, 1u);
        st_agent(&s.ctl->ovf[(c.step + 1) % 3], 1u);
    }
    if (track) {
        const int lo = wave_inclusive_sum((int) (fe & 0xFFFFu));
        const int hi = wave_inclusive_sum((int) (fe >> 16));
        if (lane_id() == kWave - 1)
            B.wfe[tid / kWave] = ((unsigned long long) (unsigned) hi << 16) + (unsigned long long) (unsigned) lo;
        __syncthreads();
        if (tid == 0) {
            unsigned long long f = 0;
            for (int w = 0; w < kWaves; w++) f += B.wfe[w];
            if (f)
                __hip_atomic_fetch_add(&s.ctl->fedges[(c.step + 1) % 3], f, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Spread step: a top-down level of few members (n <= kFastCap) with more
// edges than the fast path takes -- typically the first level after the
// source, a handful of hubs.  The tile phase would hand each row to one
// workgroup, or publish the long ones for a hub phase behind another grid
// barrier; here every workgroup loads the whole frontier into LDS, scans its
// degrees and walks an equal share of the level's edges (kBlock * kFastK at
// a time, strided over the grid), so the level is one phase and one grid
// barrier whatever its row lengths.  Each batch reserves its queue slots
// with one atomic per workgroup.  next_bits as for body_expand_contract.
// Every thread of every workgroup calls it; F must not be live.
template <bool PRED>
__device__ __forceinline__ void spread_step(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, FastFront &F,
                            StepIo io, unsigned *next_bits)
{
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int *in = s.q[c.step & 1];
    for (unsigned i = threadIdx.x; i < n; i += kBlock) {
        const int v = ld_queue(in + i);
        const int b = g.row[v];
        F.v[0][i] = v;
        F.beg[0][i] = b;
        F.deg[0][i] = g.row[v + 1] - b;
    }
    __syncthreads();
    const int total = fast_scan(F, 0, n);
    const int next_depth = c.iteration + 1;
    Control *ctl = s.ctl;
    int *out = s.q[(c.step + 1) & 1];
    int *pout = PRED ? s.pq[(c.step + 1) & 1] : nullptr;
    unsigned long long fe = 0;
    const int stride = (int) gridDim.x * kBlock * kFastK;
    for (int b0 = (int) blockIdx.x * kBlock * kFastK; b0 < total; b0 += stride) {
        int u[kFastK], pv[kFastK], ub[kFastK], ud[kFastK];
        const unsigned fresh = fast_edges<PRED, true, false>(g, s, next_depth, F.deg[0], F.beg[0], F.v[0], n, total,
                                                       b0 + (int) threadIdx.x * kFastK, u, pv, ub, ud, false, nullptr,
                                                       io);
        int got;
        const int off = block_exclusive_sum(__popc(fresh), F.scan, &got);
        // (every thread read the previous batch's base before the scan's
        // first barrier)
        if (threadIdx.x == 0 && got) F.count = add_agent(&ctl->qlen[(c.step + 1) % 3], (unsigned) got);
        __syncthreads();
        const unsigned p0 = F.count + (unsigned) off;
        bool lost = false;
#pragma unroll
        for (int k = 0; k < kFastK; k++) {
            const unsigned p = p0 + (unsigned) __popc(fresh & ((1u << k) - 1u));
            if ((fresh >> k) & 1) {
                fe += (unsigned) (ud[k] - ub[k]);
                if (p < s.cap && io.light) {
                    st_agent(out + p, u[k]);
                    if (PRED) st_agent(pout + p, pv[k]);
                } else if (p < s.cap) {
                    out[p] = u[k];
                    if (PRED) pout[p] = pv[k];
                } else {
                    lost = true;
                }
            }
        }
        if (lost) {
            st_agent(&ctl->overflow, 1u);
            st_agent(&ctl->ovf[(c.step + 1) % 3], 1u);
        }
        if (next_bits) {
#pragma unroll
            for (int k = 0; k < kFastK; k++)
                if ((fresh >> k) & 1)
                    __hip_atomic_fetch_or(next_bits + (u[k] >> 5), 1u << (u[k] & 31), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // one update per workgroup of the next frontier's edges
    const int lo = wave_inclusive_sum((int) (fe & 0xFFFFu));
    const int hi = wave_inclusive_sum((int) (fe >> 16));
    if (lane == kWave - 1) {
        F.wfe[wave] = ((unsigned long long) (unsigned) hi << 16) + (unsigned long long) (unsigned) lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long f = 0;
        for (int w = 0; w < kWaves; w++) f += F.wfe[w];
        if (s.track_edges && f)
            __hip_atomic_fetch_add(&ctl->fedges[(c.step + 1) % 3], f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// Adjacency records of low-degree graphs (lattices, road networks): every
// vertex's neighbours in one aligned record of 4 or 8 words, each the
// neighbour's number and, above it, that neighbour's degree (all ones: none),
// written once when the problem is created.  A level of the LDS path then
// costs one memory trip -- the members' records -- where it took two (column
// entries, then the claimed vertices' row bounds): the claims are LDS
// atomics, and a claimed vertex comes with its degree.  Bound: that trip, the
// one CU's line requests on wide levels, and one workgroup barrier; grid2d
// 1000^2 (1999 levels) 6.8 -> 4.0 ms, a level of tens of members 1.9 -> 1.6 us
// and of a thousand 5 -> 2.4.
// ---------------------------------------------------------------------------
constexpr int kAdjDegreeShift = 24;                 // vertices below 2^24, degrees up to 8
constexpr int kAdjMaxDegree = 8;
constexpr unsigned kAdjNone = ~0u;
static_assert(kFastVisitedWords * 32 <= (1 << kAdjDegreeShift), "a record holds the vertex number");
constexpr int kAdjCap = 3 * kFastCap;               // members kept in LDS: the frontier buffers hold numbers only
static_assert(2 * kAdjCap * sizeof(int) <= offsetof(FastFront, maxdeg), "two buffers fit the frontier arrays");

__global__ void adjacency_kernel(const int *row, const int *col, int nodes, int width, unsigned *adj)
{
    const long long count = (long long) nodes * width;
    for (long long i = blockIdx.x * (long long) blockDim.x + threadIdx.x; i < count;
         i += (long long) gridDim.x * blockDim.x) {
        const int v = (int) (i / width), e = row[v] + (int) (i % width);
        unsigned x = kAdjNone;
        if (e < row[v + 1]) {
            const int u = col[e];
            x = (unsigned) u | (unsigned) (row[u + 1] - row[u]) << kAdjDegreeShift;
        }
        adj[i] = x;
    }
}

// One level: the n members of src claim their neighbours (LDS bitmap vbits),
// label them, and append them to dst (past kAdjCap to the global queue
// `spill`).  *count and *edges, zero before, get the new members and their
// degree sum; a workgroup barrier must follow.  Every thread calls it.
template <bool PRED, int W>
__device__ __forceinline__ void adjacency_level(const SearchArgs &s, int next_depth, unsigned n, const int *src,
                                                int *dst, int *spill, unsigned *vbits, unsigned *count,
                                                unsigned *edges)
{
    constexpr int M = 8 / W;  // members per thread and round
    const unsigned wave0 = threadIdx.x & ~(unsigned) (kWave - 1);
    // (waves past the members skip the round together)
    for (unsigned base = 0; base + wave0 < n; base += M * kBlock) {
        int v[M];
        u32x4 a[M][W / 4];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const unsigned i = base + (unsigned) (m * kBlock) + threadIdx.x;
            v[m] = i < n ? src[i] : -1;
        }
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int q = 0; q < W / 4; q++) {
                a[m][q] = u32x4{kAdjNone, kAdjNone, kAdjNone, kAdjNone};
                if (v[m] >= 0)
                    a[m][q] = *reinterpret_cast<const u32x4 *>(s.adj + (size_t) v[m] * W + 4 * q);
            }
        unsigned old[8], fresh = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const unsigned x = a[k / W][(k % W) / 4][k % 4], u = x & ((1u << kAdjDegreeShift) - 1u);
            old[k] = ~0u;
            if (x != kAdjNone)
                old[k] = __hip_atomic_fetch_or(vbits + (u >> 5), 1u << (u & 31u), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        // (all claims are issued before the first result is used)
#pragma unroll
        for (int k = 0; k < 8; k++) asm volatile("" : "+v"(old[k]));
        int fe = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const unsigned x = a[k / W][(k % W) / 4][k % 4], u = x & ((1u << kAdjDegreeShift) - 1u);
            if (!((old[k] >> (u & 31u)) & 1u)) {
                fresh |= 1u << k;
                fe += (int) (x >> kAdjDegreeShift);
                s.depth[u] = next_depth;
                if (PRED) s.pred[u] = v[k / W];
            }
        }
        const int cnt = __popc(fresh);
        const int incl = wave_inclusive_sum(cnt | fe << 16);  // (at most 512 and 4096 a wave)
        const int tot = readlane(incl, kWave - 1);
        if ((tot & 0xFFFF) == 0) continue;
        unsigned at = 0;
        if (lane_id() == 0) {
            at = atomicAdd(count, (unsigned) (tot & 0xFFFF));
            atomicAdd(edges, (unsigned) (tot >> 16));
        }
        unsigned p = (unsigned) readlane((int) at, 0) + (unsigned) ((incl & 0xFFFF) - cnt);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (!((fresh >> k) & 1u)) continue;
            const int u = (int) (a[k / W][(k % W) / 4][k % 4] & ((1u << kAdjDegreeShift) - 1u));
            if (p < (unsigned) kAdjCap) dst[p] = u;
            else if (p < s.cap) spill[p] = u;
            p++;
        }
    }
}

// Runs LDS fast levels from step c (input: n <= kFastCap members in the
// global queue) until a level's output is empty, too large for the path, or
// (direction-optimizing) calls for bottom-up.  Leaves the global queue,
// counters and the fast_* hand-off exactly as the ordinary steps would have.
// `fv`: visited-edge sum through step c, fe_in: step c's frontier edges
// (see direction_rule).  Block 0 only; every thread calls it.
template <bool PRED, bool EXACT, bool FASTV>
__device__ __forceinline__ void fast_lds_path(const GraphArgs &g, const SearchArgs &s, Cursor c, unsigned n, int loop,
                              unsigned long long fv, unsigned long long fe_in, FastLds<FASTV> &L, bool wait_others)
{
    FastFront &F = L.f;
    const int *in = s.q[c.step & 1];
    // FASTV: the path's claims go to an LDS copy of the visited bitmap (no
    // other workgroup reads or writes visited words until the grid barrier
    // that ends the path); it is written back before that barrier.
    const bool ldsv = FASTV && s.nodes <= kFastVisitedWords * 32;
    const int vwords = (s.nodes + 31) >> 5;
    if (ldsv) {
        // 16-byte chunks, kLoad per thread in flight together
        constexpr int kLoad = 16;
        const u32x4 *from = reinterpret_cast<const u32x4 *>(s.visited);
        u32x4 *to = reinterpret_cast<u32x4 *>(L.vbits);
        const int chunks = vwords >> 2;
        for (int base = 0; base < chunks; base += kBlock * kLoad) {
            u32x4 t[kLoad];
#pragma unroll
            for (int j = 0; j < kLoad; j++) {
                const int i = base + j * kBlock + (int) threadIdx.x;
                if (i < chunks) t[j] = from[i];
            }
#pragma unroll
            for (int j = 0; j < kLoad; j++) {
                const int i = base + j * kBlock + (int) threadIdx.x;
                if (i < chunks) to[i] = t[j];
            }
        }
        for (int i = 4 * chunks + (int) threadIdx.x; i < vwords; i += kBlock) L.vbits[i] = s.visited[i];
    }
    int src = 0;
    unsigned long long queued = 0;
    // deepest label so far (as prepare_step notes it for the entry step)
    int maxd = c.phase == kPhaseExpandContract ? c.iteration : c.iteration - 1;
    unsigned n2 = 0;
    unsigned long long fe2 = 0;
    // frontier edges of the members and of the level before them
    unsigned long long cur_fe = fe_in, prev_fe = 0;
    const bool ce = loop == kLoopCE, tp = loop == kLoopTP;
    if (ce || tp) {
        // Contract-expand and two-phase enter at a step that contracts a
        // list of candidates (the previous level's neighbours or their
        // filtered remainder, with their parents).  Its claims, labelled
        // with the step's iteration as the step labels them, become the LDS
        // members; each level below then does the next contraction.
        // Contract-expand counts a step's input (the frontier edges of the
        // members before it) in total_queued; two-phase counts an expand
        // (the members), a filter (their edges) and a contraction (the
        // edges to vertices the level claims).
        if (threadIdx.x == 0) {
            F.count = 0;
            if (c.step < kLevelLog) {
                s.ctl->level_len[c.step] = n;
                s.ctl->level_clock[c.step] = wall_clock64();
            }
        }
        __syncthreads();
        queued += n;
        const int *pin = (c.step & 1) ? s.pq[1] : s.pq[0];
        static_assert(kFastCap <= 2 * kBlock, "two input items per thread");
        int u[2], pv[2], ub[2], ud[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const unsigned i = threadIdx.x + (unsigned) k * kBlock;
            u[k] = i < n ? ld_queue(in + i) : -1;
            pv[k] = PRED && i < n ? ld_queue(pin + i) : -1;
        }
        const unsigned fresh =
            fast_claim_vertices<PRED, EXACT, true, 2>(g, s, c.iteration, pv, u, ub, ud, ldsv, L.vbits);
        unsigned long long fe = 0;
        bool labeled = false;
        int dmax = 0;
        fast_append<2>(s, F, 0, (c.step & 1) ? s.q[0] : s.q[1], fresh, u, ub, ud, fe, labeled, dmax);
        fast_fold(F, 0, fe, labeled, dmax);
        n = F.count;  // (at most the input's n <= kFastCap: nothing spilled)
        fe2 = F.fe;
        if (F.labeled) maxd = c.iteration;
        if (n == 0) c = advance(loop, c);  // the next step's input is empty
    } else {
        int dmax = 0;
        for (unsigned i = threadIdx.x; i < n; i += kBlock) {
            const int v = ld_queue(in + i);
            const int b = g.row[v];
            const int d = g.row[v + 1] - b;
            F.v[0][i] = v;
            F.beg[0][i] = b;
            F.deg[0][i] = d;
            dmax = max(dmax, d);
        }
        dmax = wave_inclusive_max_nonneg(dmax);
        if (lane_id() == kWave - 1) F.wmax[threadIdx.x / kWave] = dmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            int dm = 0;
            for (int w = 0; w < kWaves; w++) dm = max(dm, F.wmax[w]);
            F.maxdeg[0] = dm;
        }
        __syncthreads();
    }
    // Adjacency levels (see above): members' numbers only, in two buffers over
    // the frontier arrays; one workgroup barrier a level, with three sets of
    // counters (a level's set was last read before the level before it).
    const bool adjacent = EXACT && FASTV && !tp && ldsv && s.adj != nullptr;
    int *abuf = &F.v[0][0];
    unsigned *acount = reinterpret_cast<unsigned *>(F.scan), *aedges = reinterpret_cast<unsigned *>(F.wmax);
    int acur = 0;
    if (adjacent) {
        __syncthreads();
        if (threadIdx.x < 3) {
            acount[threadIdx.x] = 0u;
            aedges[threadIdx.x] = 0u;
        }
        __syncthreads();
        const unsigned most = (unsigned) min((long long) kAdjCap, 3ll * s.fast_t);
        int set = 0;
        while (n > 0) {
            const int logged = c.step + (ce ? 1 : 0);
            const unsigned long long step_input = ce ? fe2 : n;
            if (threadIdx.x == 0 && logged < kLevelLog) {
                s.ctl->level_len[logged] = (unsigned) step_input;
                s.ctl->level_clock[logged] = wall_clock64();
            }
            queued += step_input;
            const int after = set == 2 ? 0 : set + 1;
            if (threadIdx.x == 0) {
                acount[after] = 0u;
                aedges[after] = 0u;
            }
            const int *from = abuf + acur * kAdjCap;
            int *to = abuf + (acur ^ 1) * kAdjCap;
            if (s.adj_width == 4)
                adjacency_level<PRED, 4>(s, c.iteration + 1, n, from, to, s.q[(c.step + 1) & 1], L.vbits,
                                         acount + set, aedges + set);
            else
                adjacency_level<PRED, 8>(s, c.iteration + 1, n, from, to, s.q[(c.step + 1) & 1], L.vbits,
                                         acount + set, aedges + set);
            __syncthreads();
            n2 = acount[set];
            fe2 = aedges[set];
            if (n2 > 0) maxd = c.iteration + 1;
            acur ^= 1;
            set = after;
            c = advance(loop, c);
            bool go = n2 > 0 && n2 <= most;
            if (go && loop == kLoopDO) {
                const unsigned long long fv2 = fv + fe2;
                if (direction_rule(s, c.phase, fe2, n2, fv2, cur_fe) != c.phase) go = false;
                else fv = fv2;
            }
            prev_fe = cur_fe;
            cur_fe = fe2;
            if (go && ce && s.sat_t >= 0 && fe2 > (unsigned long long) s.sat_t) go = false;
            n = n2;
            if (!go) break;
        }
    }
    while (!adjacent && n > 0) {
        // Two-phase counts a contraction's input -- every edge the filter
        // passes, i.e. every edge to a vertex the level claims -- which
        // direct levels count; the grid takes the others.
        if (tp && !fast_direct(F.maxdeg[src], n)) {
            n2 = n;
            break;
        }
        // (a contract-expand level is the contraction of step c + 1)
        const int logged = c.step + (ce ? 1 : 0);
        const unsigned long long step_input = ce ? fe2 : tp ? n + fe2 : n;
        if (threadIdx.x == 0 && logged < kLevelLog) {
            s.ctl->level_len[logged] = (unsigned) step_input;
            s.ctl->level_clock[logged] = wall_clock64();
        }
        queued += step_input;
        // the queue the step after the path reads if this level ends it
        // (members past kFastCap go there): that of step c + 1, or of the
        // expand step four steps on from a two-phase contraction
        int *spill = tp ? s.q[c.step & 1] : s.q[(c.step + 1) & 1];
        fast_lds_level<PRED, EXACT>(g, s, c, n, src, F, ldsv, L.vbits, spill, tp);
        n2 = F.count;
        fe2 = F.fe;
        if (F.labeled) maxd = c.iteration + 1;
        src ^= 1;
        c = advance(loop, c);
        if (tp) {
            // expand and filter, then the contraction of the filter's output
            queued += (unsigned long long) n2 + F.dups;
            c = advance(loop, advance(loop, c));
        }
        bool go = n2 > 0 && n2 <= (unsigned) kFastCap && n2 <= (unsigned) s.fast_t && fe2 <= kFastEdges;
        if (go && loop == kLoopDO) {
            const unsigned long long fv2 = fv + fe2;
            if (direction_rule(s, c.phase, fe2, n2, fv2, cur_fe) != c.phase) go = false;
            else fv = fv2;
        }
        prev_fe = cur_fe;
        cur_fe = fe2;
        // a hybrid search leaves contract-expand when a step's input
        // exceeds the saturation threshold: the grid takes that step
        if (go && ce && s.sat_t >= 0 && fe2 > (unsigned long long) s.sat_t) go = false;
        n = n2;
        if (!go) break;
        __syncthreads();  // every thread has read F's results before the next level resets them
    }
    // Contract-expand hands its members to the grid as the input of an
    // expand step (cursor c, phase expand: their neighbours become step
    // c + 1's edge frontier), whose input the loop top adds to total_queued
    // although it is not a contract-expand step's.
    if (ce && n2 > 0) {
        c.phase = kPhaseExpand;
        queued -= min(n2, s.cap);
    }
    // Two-phase hands its members to the expand step after their
    // contraction, which counts them as its input.
    if (tp && n2 > 0) c = advance(loop, c);
    if (ldsv) {
        // (the last level's claims precede its closing workgroup barrier)
        const u32x4 *from = reinterpret_cast<const u32x4 *>(L.vbits);
        u32x4 *to = reinterpret_cast<u32x4 *>(s.visited);
        const int chunks = vwords >> 2;
        for (int i = threadIdx.x; i < chunks; i += kBlock) to[i] = from[i];
        for (int i = 4 * chunks + (int) threadIdx.x; i < vwords; i += kBlock) s.visited[i] = L.vbits[i];
    }
    // The hand-off below rewrites counters the other workgroups may still
    // be reading at the top of the step the path started from, unless they
    // have all arrived at the barrier that ends the path.
    if (wait_others) {
        if (threadIdx.x == 0) wait_other_arrivals(s.ctl);
        __syncthreads();
    }
    // The next step (c) reads its input from the global queue: copy the
    // LDS-resident members (those past kFastCap were written there already).
    const unsigned held = min(n2, (unsigned) (adjacent ? kAdjCap : kFastCap));
    const int *members = adjacent ? abuf + acur * kAdjCap : F.v[src];
    int *q = s.q[c.step & 1];
    for (unsigned i = threadIdx.x; i < held && i < s.cap; i += kBlock) q[i] = members[i];
    if (threadIdx.x == 0) {
        Control *ctl = s.ctl;
        // what the previous step's prepare_step would have left for step c
        st_agent(&ctl->qlen[(c.step + 1) % 3], 0u);
        st_agent(&ctl->steal[c.step & 1], 0u);
        st_agent(&ctl->hub_steal[c.step & 1], 0u);
        st_agent(&ctl->compact, 0u);
        st_agent(&ctl->ovf[(c.step + 1) % 3], 0u);
        __hip_atomic_store(&ctl->hub_alloc[c.step & 1], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctl->fedges[(c.step + 1) % 3], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // step c's input
        st_agent(&ctl->qlen[c.step % 3], min(n2, s.cap));
        st_agent(&ctl->ovf[c.step % 3], n2 > s.cap ? 1u : 0u);
        if (n2 > s.cap) st_agent(&ctl->overflow, 1u);
        __hip_atomic_store(&ctl->fedges[c.step % 3], fe2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (maxd >= 0) atomicMax(&ctl->max_depth, maxd);
        __hip_atomic_fetch_add(&ctl->total_queued, queued, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        st_agent(&ctl->fast_step, c.step);
        st_agent(&ctl->fast_iteration, c.iteration);
        st_agent(&ctl->fast_phase, c.phase);
        // excludes the step the loop top runs next (it adds it)
        __hip_atomic_store(&ctl->fast_vsum, fv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctl->fast_prev_fe, prev_fe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// Search start and end inside a persistent launch (one launch per search).
// ---------------------------------------------------------------------------

// Every workgroup rewrites its share of the labels (with init_reset); block 0
// clears the status head and the level log and queues the source.  Only the
// labels and block 0's own words are written, so the first step may begin
// before a grid barrier as long as it reads nothing of the control block
// and claims nothing before one (the loop top takes step 0's values from
// search_start_values).
__device__ __forceinline__ void search_prologue(const GraphArgs &g, const SearchArgs &s, bool clear_bitmaps)
{
    const int src = s.init_src;
    if (clear_bitmaps) {
        // both frontier bitmaps, which are contiguous
        const int words = 2 * ((s.nodes + 31) >> 5);
        for (int i = blockIdx.x * kBlock + threadIdx.x; i < words; i += gridDim.x * kBlock) s.fbm[0][i] = 0u;
    }
    if (s.init_reset) {
        const int words = (s.nodes + 31) >> 5;
        for (int i = blockIdx.x * kBlock + threadIdx.x; i < s.nodes; i += gridDim.x * kBlock) {
            const bool is_src = s.init_label && i == src;
            s.depth[i] = is_src ? 0 : -1;
            if (s.pred) s.pred[i] = is_src ? -2 : -1;
            if (i < words) s.visited[i] = (s.init_label && (src >> 5) == i) ? 1u << (src & 31) : 0u;
        }
    }
    if (blockIdx.x != 0) return;
    Control *ctl = s.ctl;
    unsigned *head = reinterpret_cast<unsigned *>(ctl);
    for (int i = threadIdx.x; i < (int) (kControlHead / 4); i += kBlock) head[i] = 0u;
    for (int i = threadIdx.x; i < kLevelLog; i += kBlock) {
        ctl->level_len[i] = 0u;
        ctl->level_clock[i] = 0ull;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        ctl->qlen[0] = 1;
        ctl->max_depth = -1;
        s.q[0][0] = src;
        if (s.pq[0]) s.pq[0][0] = -2;
        if (s.init_label) {
            if (!s.init_reset) {
                s.depth[src] = 0;
                if (s.pred) s.pred[src] = -2;
                s.visited[src >> 5] |= 1u << (src & 31);
            }
            ctl->max_depth = 0;
            const unsigned long long deg = (unsigned long long) (g.row[src + 1] - g.row[src]);
            ctl->fedges[0] = deg;
        }
    }
}

// Block 0 copies the status head to s.host_head when the level loop ends,
// so the host reads it after the launch without a copy of its own.  The
// loop ends at a loop top, after the grid barrier that completed the last
// step's counter updates, and the exit fields are block 0's own: the head
// is final (the instrumented cycle sums, added later, are not copied).
// Called by thread 0 of block 0.
__device__ __forceinline__ void publish_status(const SearchArgs &s)
{
    const unsigned *head = reinterpret_cast<const unsigned *>(s.ctl);
    unsigned *out = reinterpret_cast<unsigned *>(s.host_head);
    unsigned w[kControlHead / 4];
#pragma unroll
    for (int i = 0; i < (int) (kControlHead / 4); i++) w[i] = __hip_atomic_load(head + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < (int) (kControlHead / 4); i++) out[i] = w[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");  // system scope: the host reads it next
}

// ---------------------------------------------------------------------------
// Persistent level loop (cooperative launch).
// ---------------------------------------------------------------------------
// One instantiation per strategy (LOOP), so profiles attribute time to the
// strategy and the level loop carries no dead strategy branches.
// Most work (frontier edges, or items when edges are not tracked) of a step
// that ends in a light barrier: up to here a step is bound by its chain of
// memory trips, past it the stores past the L2 and the row reads beside the
// claims would cost more than the cache maintenance they replace.
constexpr unsigned long long kLightWork = 1ull << 19;

// Work of a step over n items whose edges are not tracked: a filtering
// expansion reads a visited word for each of its members' edges, past the L2
// in a light step, about as many as the graph's vertices have.
__device__ __forceinline__ unsigned long long item_work(const SearchArgs &s, int phase, unsigned n)
{
    if (phase != kPhaseExpand || !filters(s)) return n;
    return (unsigned long long) n * (s.total_edges / (unsigned long long) s.nodes + 1);
}

template <bool PRED, bool EXACT, int LOOP, bool FASTV>
__global__ __launch_bounds__(kBlock) void persistent_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    constexpr int loop = LOOP;
    __shared__ LoopLds<PRED, FASTV> shared;
    Lds<PRED> &lds = shared.step;
    init_lds(lds);
    unsigned long long t_begin = s.instrument ? wall_clock64() : 0, busy = 0;
    int reason = kExitDone;
    // Visited-edge sum up to the current step, kept by every workgroup from
    // counters that no workgroup changes during the step (fedges[step % 3])
    // -- see direction_rule.  fedges[0] holds the source's degree.
    unsigned long long vsum = 0;
    // the previous step's frontier edges (direction rule; grid-uniform too)
    unsigned long long prev_fe = 0;

    // With a folded search start, step 0's loop-top values come from the
    // graph (one source, its degree), not from the control block that block
    // 0 is still writing, and the step's first grid barrier orders the
    // label rewrite before any claim.
    bool start = s.init_src >= 0;
    // Barriers: full ones order plain stores before plain loads; light ones
    // (after light steps, see StepIo) only what goes past the XCDs' L2s, and
    // leave the caches stale: the next step that is not light itself
    // refreshes them first.  Searches with best-effort contractions read
    // labels, which are plain stores, so their barriers are all full.
    bool stale = false;
    auto bar = [&](bool light) {
        if (EXACT && light) {
            grid_barrier_light(s.ctl);
            stale = true;
        } else {
            grid_barrier(s.ctl);
            stale = false;
        }
    };
    auto refresh = [&]() {
        if (stale) refresh_caches();
        stale = false;
    };
    if (start) search_prologue(g, s, LOOP == kLoopDO);
    // Frontier bitmaps of a direction-optimizing loop (grid-uniform state):
    // which are not known to be clear, and the step whose frontier one of
    // them holds exactly (written by a marked step's compaction).
    unsigned fbm_dirty = start ? 0u : 3u;
    int fbm_exact_step = -1;

    // Every decision at the top of a step reads only values final before
    // the step began and unchanged during it (the input length, the
    // previous step's overflow flag, this step's frontier edges), so all
    // workgroups take the same branch and meet the same grid barriers.
    while (true) {
        unsigned n;
        unsigned long long fe = 0;
        bool bu_exit = false;  // bottom-up until this step
        if (start) {
            n = 1;
            if (s.track_edges && s.init_label) fe = (unsigned long long) (g.row[s.init_src + 1] - g.row[s.init_src]);
        } else {
            n = frontier_length(s, c.step);
            if (ld_agent(&s.ctl->ovf[c.step % 3])) { reason = kExitOverflow; break; }
            if (n == 0) { reason = kExitDone; break; }
            if (s.track_edges) fe = ld64_agent(&s.ctl->fedges[c.step % 3]);
        }
        // (an expand step that ends a contract-expand fast path runs first)
        if (loop == kLoopCE && c.phase != kPhaseExpand && s.sat_t >= 0 && n > (unsigned) s.sat_t) {
            reason = kExitSaturated;
            break;
        }
        if (loop == kLoopDO) {
            vsum += fe;
            int dir = direction_rule(s, c.phase, fe, n, vsum, prev_fe);
            prev_fe = fe;
            if (start && dir != c.phase) {
                bar(false);
                start = false;
            }
            if (dir == kPhaseBottomUp) refresh();
            if (dir == kPhaseBottomUp && c.phase != kPhaseBottomUp) {
                if (fbm_exact_step != c.step) {
                    if (fbm_dirty & (1u << (c.iteration & 1))) {
                        frontier_bitmap_pass(g, s, c, n, 0);
                        bar(false);
                    }
                    frontier_bitmap_pass(g, s, c, n, 1);
                    bar(false);
                }
                fbm_dirty = 3u;  // bottom-up levels write both
            } else if (dir != kPhaseBottomUp && c.phase == kPhaseBottomUp) {
                bu_exit = true;
            }
            c.phase = dir;
        }

        // Contract-expand and two-phase take the LDS path from a step that
        // contracts at most kFastCap items (never from the expand step the
        // path hands over to the grid with).
        const bool contract_lds = ((LOOP == kLoopCE && c.phase == kPhaseContractExpand) ||
                                   (LOOP == kLoopTP && c.phase == kPhaseContract)) &&
                                  n <= (unsigned) kFastCap;
        // Two-phase expand steps always take the grid: one workgroup alone
        // also costs an entry barrier, and their rows may be long (a 1 M-vertex
        // random tree 943 -> 900 us, R-MAT scale 15 186 -> 155 us).
        const bool fast = fast_level(s, c, n, fe) && gridDim.x > 1 && !(LOOP == kLoopCE && c.phase == kPhaseExpand) &&
                          (LOOP != kLoopTP || c.phase == kPhaseContract) &&
                          ((LOOP != kLoopEC && LOOP != kLoopDO) || (n <= (unsigned) kFastCap && fe <= kFastEdges));
        // large top-down levels mark instead of claiming (grid-uniform: fe
        // is this step's frontier-edge count); few-member ones spread their
        // edges over the grid
        const bool mark =
            (LOOP == kLoopEC || LOOP == kLoopDO) && c.phase == kPhaseExpandContract && marked_step(s, fe);
        // large steps of graphs with an LDS bitmap take bit marks instead
        // (contractions chained through tile status words keep their order)
        // (few members keep the spread form up to the byte marks' rule)
        const bool bits =
            FASTV && !fast &&
            ((LOOP == kLoopEC || LOOP == kLoopDO)
                 ? c.phase == kPhaseExpandContract && (mark || n > (unsigned) kFastCap) && bit_step(s, fe)
             : LOOP == kLoopTP ? c.phase == kPhaseContract && !s.tile_status && bit_step(s, n)
                               : c.phase == kPhaseContractExpand && bit_step(s, n));
        const bool spread = (LOOP == kLoopEC || LOOP == kLoopDO) && c.phase == kPhaseExpandContract && !mark &&
                            n <= (unsigned) kFastCap && s.spread;
        // The first top-down step after bottom-up levels reads its frontier
        // from the bitmap they left, unless its form needs the queue (the
        // fast path, spread and marked steps index it).
        const bool from_bitmap = bu_exit && !fast && !mark && !bits && !spread;
        if (bu_exit && !from_bitmap) {
            queue_from_bitmap<PRED>(g, s, c, lds);  // clears both bitmaps
            bar(false);
            fbm_dirty = 0u;
        }
        if (start && !fast) bar(false);
        const bool first = start;
        start = false;
        if (fast) {
            // Single-workgroup fast path: block 0 runs consecutive small
            // levels with workgroup barriers only (no grid tier: it alone
            // works); the rest of the grid waits at the next grid barrier.
            // Every workgroup must be done reading this step's counters
            // before block 0 rewrites them (its second fast step zeroes
            // qlen / fedges of index step % 3, which a workgroup still on
            // its way out of the previous barrier would otherwise read as an
            // empty frontier and leave the loop, stranding the grid at the
            // barrier below).  The per-level path rewrites counters as it
            // goes and takes an entry barrier.  The LDS path writes them
            // only when it ends, so it starts at once and, before writing,
            // waits for the others' arrival at the closing barrier -- except
            // after a folded search start, whose label rewrite the entry
            // barrier orders before the first claim.
            const bool lds_path = LOOP == kLoopEC || LOOP == kLoopDO || contract_lds;
            if (!lds_path || first) bar(!first);
            if (lds_path) {
                // frontier kept in LDS between levels
                if (blockIdx.x == 0) {
                    unsigned long long t0 = s.instrument ? wall_clock64() : 0;
                    refresh();
                    fast_lds_path<PRED, EXACT, FASTV>(g, s, c, n, loop, vsum, fe, shared.fast, lds_path && !first);
                    release_caches();
                    __syncthreads();
                    init_lds(lds);
                    if (s.instrument) busy += wall_clock64() - t0;
                }
            } else if (blockIdx.x == 0) {
                unsigned long long t0 = s.instrument ? wall_clock64() : 0;
                unsigned long long fv = vsum;  // sum through the step being run
                refresh();
                // (the step bodies grab every tile: see tile_grab)
                if (threadIdx.x == 0) lds.solo = 1;
                __syncthreads();
                while (true) {
                    if (threadIdx.x == 0) prepare_step(s.ctl, c, n);
                    loop_body<PRED, EXACT, LOOP>(c.phase, g, s, c, n, lds, 0, false, 0ull, StepIo{false, false});
                    // the next level reads queue entries other waves just
                    // stored: each wave's stores must have completed, which
                    // __syncthreads() alone does not wait for
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
                    c = advance(loop, c, LOOP == kLoopTP && filters(s));
                    if (threadIdx.x == 0) lds.nb = frontier_length(s, c.step);
                    __syncthreads();
                    n = lds.nb;
                    if (n == 0 || !fast_level(s, c, n) || ld_agent(&s.ctl->ovf[c.step % 3])) break;
                    if (loop == kLoopCE && s.sat_t >= 0 && n > (unsigned) s.sat_t) break;
                    // (a small two-phase contraction is the LDS path's entry)
                    if (loop == kLoopTP && c.phase == kPhaseContract && n <= (unsigned) kFastCap) break;
                    // (direction-optimizing searches always take the LDS path)
                }
                if (threadIdx.x == 0) {
                    st_agent(&s.ctl->fast_step, c.step);
                    st_agent(&s.ctl->fast_iteration, c.iteration);
                    st_agent(&s.ctl->fast_phase, c.phase);
                    // excludes the step the loop top runs next (it adds it)
                    __hip_atomic_store(&s.ctl->fast_vsum, fv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    lds.solo = 0;  // (the grid barrier below orders it)
                }
                release_caches();
                if (s.instrument) busy += wall_clock64() - t0;
            }
            bar(true);  // (block 0 alone wrote anything, and has written its L2 back)
            c.step = ld_agent(&s.ctl->fast_step);
            c.iteration = ld_agent(&s.ctl->fast_iteration);
            c.phase = ld_agent(&s.ctl->fast_phase);
            vsum = ld64_agent(&s.ctl->fast_vsum);
            prev_fe = ld64_agent(&s.ctl->fast_prev_fe);
            continue;
        }

        unsigned long long t0 = s.instrument ? wall_clock64() : 0;
        // A top-down step of a direction-optimizing search marks its claims
        // in the next frontier's bitmap when that bitmap is clear, so a turn
        // to bottom-up after it needs no bitmap pass.
        unsigned *next_bits = nullptr;
        if (LOOP == kLoopDO && !mark && c.phase == kPhaseExpandContract &&
            !(fbm_dirty & (1u << ((c.iteration + 1) & 1)))) {
            next_bits = s.fbm[(c.iteration + 1) & 1];
            fbm_dirty |= 1u << ((c.iteration + 1) & 1);
            fbm_exact_step = c.step + 1;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) prepare_step(s.ctl, c, n);
        const bool light_step = EXACT && c.phase != kPhaseBottomUp && !mark && !bits && !from_bitmap &&
                                (LOOP == kLoopTP ? item_work(s, c.phase, n) : s.track_edges ? fe : (unsigned long long) n) <= kLightWork;
        if (!light_step) refresh();
        const StepIo io{light_step, stale};
        if (bits) {
            if constexpr (FASTV) {
                BitLds &B = *reinterpret_cast<BitLds *>(&shared.fast.f);
                unsigned *vbits = shared.fast.vbits;
                __syncthreads();
                bits_clear(s, vbits);
                if constexpr (LOOP == kLoopEC || LOOP == kLoopDO) {
                    bits_from_rows<PRED>(g, s, c, n, B, vbits);
                    if (s.max_degree >= min(s.grid_t, kWaveHubRow)) {
                        bar(true);
                        refresh();  // (the list is read through the caches)
                        bits_from_hubs<PRED>(g, s, c, vbits);
                    }
                } else {
                    bits_from_items<PRED, EXACT>(s, c, n, vbits);
                }
                bits_dump(s, vbits);
                if (s.instrument) busy += wall_clock64() - t0;
                bar(true);
                t0 = s.instrument ? wall_clock64() : 0;
                unsigned *fbm_out = nullptr;
                if (LOOP == kLoopDO) {
                    fbm_out = s.fbm[(c.iteration + 1) & 1];
                    fbm_dirty |= 1u << ((c.iteration + 1) & 1);
                    fbm_exact_step = c.step + 1;
                }
                refresh();  // (slabs and visited words are read plainly)
                // (what others read next goes past the L2 and a light barrier
                // follows: R-MAT scale 19 expand-contract 244 -> 235 us)
                const bool through = EXACT;
                if (LOOP == kLoopEC || LOOP == kLoopDO)
                    bits_collect<EXACT>(g, s, c, c.iteration + 1, B, s.q[(c.step + 1) & 1],
                                        &s.ctl->qlen[(c.step + 1) % 3], fbm_out, s.track_edges != 0, through);
                else if (LOOP == kLoopTP)
                    bits_collect<EXACT>(g, s, c, c.iteration, B, s.q[(c.step + 1) & 1],
                                        &s.ctl->qlen[(c.step + 1) % 3], nullptr, false, through);
                else  // (the input is spent: its queue takes the members)
                    bits_collect<EXACT>(g, s, c, c.iteration, B, s.q[c.step & 1], &s.ctl->compact, nullptr, false,
                                        through);
                __syncthreads();
                init_lds(lds);
                if (s.instrument) busy += wall_clock64() - t0;
                bar(through);
                if constexpr (LOOP == kLoopCE) {
                    // the members expand into the next edge frontier
                    const unsigned m = ld_agent(&s.ctl->compact);
                    const StepIo xio{false, false};
                    if (m > 0) {
                        if (blockIdx.x == 0 && threadIdx.x == 0) atomicMax(&s.ctl->max_depth, c.iteration);
                        t0 = s.instrument ? wall_clock64() : 0;
                        refresh();
                        body_expand<PRED, EXACT>(g, s, c, m, lds, 0, true, xio);
                        if (s.instrument) busy += wall_clock64() - t0;
                        bar(false);
                        if (s.max_degree >= min(s.grid_t, kHeavyRowNarrow) && hubs_pending(s, c.step)) {
                            t0 = s.instrument ? wall_clock64() : 0;
                            body_expand<PRED, EXACT>(g, s, c, m, lds, 1, true, xio);
                            if (s.instrument) busy += wall_clock64() - t0;
                            bar(false);
                        }
                    }
                }
            }
            c = advance(loop, c);
            continue;
        }
        if (spread) {
            if constexpr (LOOP == kLoopEC || LOOP == kLoopDO) {
                spread_step<PRED>(g, s, c, n, shared.fast.f, io, next_bits);
                __syncthreads();
                init_lds(lds);
            }
        } else if (mark) {
            body_expand_mark<PRED>(g, s, c, n, lds, 0, true);
        } else {
            loop_body<PRED, EXACT, LOOP>(c.phase, g, s, c, n, lds, 0, true, fe, io, next_bits, from_bitmap);
        }
        if (s.instrument) busy += wall_clock64() - t0;
        bar(light_step);
        // (graphs whose longest row no step publishes have no list to look at)
        if (!spread && gathers(c.phase) && s.max_degree >= min(s.grid_t, kHeavyRowNarrow) && hubs_pending(s, c.step)) {
            t0 = s.instrument ? wall_clock64() : 0;
            refresh();  // (the list is read through the caches)
            const StepIo io{light_step, false};
            if (mark) body_expand_mark<PRED>(g, s, c, n, lds, 1, true);
            else loop_body<PRED, EXACT, LOOP>(c.phase, g, s, c, n, lds, 1, true, fe, io, next_bits, from_bitmap);
            if (s.instrument) busy += wall_clock64() - t0;
            bar(light_step);
        }
        if (mark) {
            t0 = s.instrument ? wall_clock64() : 0;
            unsigned *fbm_out = nullptr;
            if (LOOP == kLoopDO) {
                fbm_out = s.fbm[(c.iteration + 1) & 1];
                fbm_dirty |= 1u << ((c.iteration + 1) & 1);
                fbm_exact_step = c.step + 1;
            }
            mark_compact<PRED>(g, s, c, lds, fbm_out);
            if (s.instrument) busy += wall_clock64() - t0;
            bar(false);
        }
        // (fbm_dirty kept this step's claims out of the bitmap it cleared)
        if (from_bitmap) fbm_dirty = 0u;
        c = advance(loop, c, LOOP == kLoopTP && filters(s));
    }

    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s.ctl->exit_reason = reason;
        s.ctl->exit_step = c.step;
        s.ctl->exit_iteration = c.iteration;
        s.ctl->exit_phase = c.phase;
        // (agent-scope loads of the words this block stored plainly)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        if (s.host_head) publish_status(s);
    }
    if (s.instrument && threadIdx.x == 0) {
        unsigned long long life = wall_clock64() - t_begin;
        atomicAdd(&s.ctl->busy_cycles, busy);
        atomicAdd(&s.ctl->life_cycles, life);
    }
}

// ---------------------------------------------------------------------------
// Launches per step: the tile phase, then (for gathering phases) the hub
// phase as its own launch.
// ---------------------------------------------------------------------------

// The step's input length n, or false when the launch has nothing to do
// (grid-uniform: every workgroup sees the same counters).
template <int PHASE>
__device__ __forceinline__ bool step_begins(const SearchArgs &s, Cursor c, unsigned &n)
{
    if (s.hybrid_steps && ld_agent(&s.ctl->hybrid_stop)) return false;
    n = frontier_length(s, c.step);
    if (ld_agent(&s.ctl->overflow)) n = 0;
    if (PHASE == kPhaseContract && s.hybrid_steps && n > 0 && n <= (unsigned) s.sat_t) {
        // The filtered edge frontier fits the persistent kernel again: it
        // runs this step (enactor_hybrid.cuh:386-532 leaves the two-phase
        // loop at the same point).  Every workgroup sees the same n.
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            s.ctl->exit_step = c.step;
            s.ctl->exit_iteration = c.iteration;
            st_agent(&s.ctl->hybrid_stop, 1u);
        }
        return false;
    }
    return true;
}

template <bool PRED, bool EXACT, int PHASE>
__global__ __launch_bounds__(kBlock) void step_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    __shared__ Lds<PRED> lds;
    unsigned n;
    if (!step_begins<PHASE>(s, c, n)) return;
    // (the step's frontier edges; a bottom-up step's are read for the sum alone)
    const unsigned long long fe = PHASE == kPhaseExpandContract || PHASE == kPhaseBottomUp
                                      ? ld64_agent(&s.ctl->fedges[c.step % 3])
                                      : 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        prepare_step(s.ctl, c, n);
        s.ctl->visited_edges += fe;  // (the host's direction rule reads it)
    }
    if (n == 0) return;
    init_lds(lds);
    run_body<PRED, EXACT>(PHASE, g, s, c, n, lds, 0, true, fe);
}

template <bool PRED, bool EXACT, int PHASE>
__global__ __launch_bounds__(kBlock) void hub_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    __shared__ Lds<PRED> lds;
    if (s.hybrid_steps && ld_agent(&s.ctl->hybrid_stop)) return;
    if (!hubs_pending(s, c.step)) return;
    init_lds(lds);
    run_body<PRED, EXACT>(PHASE, g, s, c, frontier_length(s, c.step), lds, 1, true, 0ull);
}

// Contract steps of graphs with bit-mark slabs: large ones set bits here and
// are collected by the launch that follows, on the same grid.
template <bool PRED, bool EXACT>
__global__ __launch_bounds__(kBlock) void contract_bits_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    __shared__ LoopLds<PRED, true> shared;
    unsigned n;
    if (!step_begins<kPhaseContract>(s, c, n)) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) prepare_step(s.ctl, c, n);
    if (n == 0) return;
    if (bit_step(s, n)) {
        bits_clear(s, shared.fast.vbits);
        bits_from_items<PRED, EXACT>(s, c, n, shared.fast.vbits);
        bits_dump(s, shared.fast.vbits);
    } else {
        init_lds(shared.step);
        body_contract<PRED, EXACT>(g, s, c, n, shared.step, StepIo{false, false});
    }
}

template <bool EXACT>
__global__ __launch_bounds__(kBlock) void contract_collect_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    __shared__ BitLds B;
    if (s.hybrid_steps && ld_agent(&s.ctl->hybrid_stop)) return;
    const unsigned n = ld_agent(&s.ctl->overflow) ? 0u : frontier_length(s, c.step);
    if (n == 0 || !bit_step(s, n)) return;
    bits_collect<EXACT>(g, s, c, c.iteration, B, s.q[(c.step + 1) & 1], &s.ctl->qlen[(c.step + 1) % 3], nullptr, false);
}

__global__ __launch_bounds__(kBlock) void frontier_bitmap_kernel(GraphArgs g, SearchArgs s, Cursor c, int pass)
{
    frontier_bitmap_pass(g, s, c, frontier_length(s, c.step), pass);
}

__global__ __launch_bounds__(kBlock) void queue_from_bitmap_kernel(GraphArgs g, SearchArgs s, Cursor c)
{
    __shared__ Lds<false> lds;
    queue_from_bitmap<false>(g, s, c, lds);
}

// ---------------------------------------------------------------------------
// Initialisation kernels.
// ---------------------------------------------------------------------------
__global__ void reset_labels_kernel(int *depth, int *pred, unsigned *visited, int nodes)
{
    int words = (nodes + 31) >> 5;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nodes; i += gridDim.x * blockDim.x) {
        depth[i] = -1;
        if (pred) pred[i] = -1;
        if (i < words) visited[i] = 0u;
    }
}

// Seeds the search: counters to zero, the source in queue 0 (predecessor -2),
// and for vertex-frontier strategies the source already labelled.  Resetting
// every counter here, before the first step, replaces the reference's
// iteration-0 counter reset inside every CTA (contract_expand_atomic/
// kernel.cuh:307-332), which can race with CTA 0's first enqueue.
// Starts a search: clears the control block, queues the source and, with
// reset set, rewrites every label in the same pass (each element written by
// exactly one thread, the source's with its start values), saving a launch.
__global__ void init_search_kernel(SearchArgs s, const int *row, int src, int label_source, int reset)
{
    if (reset) {
        const int words = (s.nodes + 31) >> 5;
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < s.nodes; i += gridDim.x * blockDim.x) {
            const bool is_src = label_source && i == src;
            s.depth[i] = is_src ? 0 : -1;
            if (s.pred) s.pred[i] = is_src ? -2 : -1;
            if (i < words) {
                const bool holds = label_source && (src >> 5) == i;
                s.visited[i] = holds ? 1u << (src & 31) : 0u;
            }
        }
    }
    if (blockIdx.x != 0) return;
    Control *ctl = s.ctl;
    unsigned *words = reinterpret_cast<unsigned *>(ctl);
    for (int i = threadIdx.x; i < (int) (sizeof(Control) / 4); i += blockDim.x) words[i] = 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
        ctl->qlen[0] = 1;
        ctl->max_depth = -1;
        s.q[0][0] = src;
        if (s.pq[0]) s.pq[0][0] = -2;
        if (label_source) {
            if (!reset) {
                s.depth[src] = 0;
                if (s.pred) s.pred[src] = -2;
                s.visited[src >> 5] |= 1u << (src & 31);
            }
            ctl->max_depth = 0;
            unsigned long long deg = (unsigned long long) (row[src + 1] - row[src]);
            ctl->fedges[0] = deg;
        }
    }
}

// ---------------------------------------------------------------------------
// Barrier microbenchmark and primitive self-test.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void barrier_bench_kernel(Control *ctl, int iterations)
{
    for (int i = 0; i < iterations; i++) grid_barrier(ctl);
}

}  // namespace b40c_hip

// Plain 16-byte-vector streaming copy (counter calibration).
extern "C" __global__ __launch_bounds__(256) void b40c_calibration_copy_kernel(const uint4 *src, uint4 *dst,
                                                                              size_t n)
{
    for (size_t i = blockIdx.x * (size_t) blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x)
        dst[i] = src[i];
}

namespace b40c_hip {

__global__ __launch_bounds__(kWave) void wave_selftest_kernel(const int *in, int *out_scan, int *out_rank, int n)
{
    int i = blockIdx.x * kWave + threadIdx.x;
    int x = i < n ? in[i] : 0;
    int s = wave_inclusive_sum(x);
    uint64_t m = ballot((x & 1) != 0);
    int r = lanes_below(m);
    if (i < n) {
        out_scan[i] = s;
        out_rank[i] = r;
    }
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
namespace {

template <bool PRED, bool EXACT>
const void *persistent_ptr(int loop, bool fastv)
{
    switch (loop) {
    case kLoopEC:
        return fastv ? reinterpret_cast<const void *>(&persistent_kernel<PRED, true, kLoopEC, true>)
                     : reinterpret_cast<const void *>(&persistent_kernel<PRED, true, kLoopEC, false>);
    case kLoopCE:
        return fastv ? reinterpret_cast<const void *>(&persistent_kernel<PRED, EXACT, kLoopCE, true>)
                     : reinterpret_cast<const void *>(&persistent_kernel<PRED, EXACT, kLoopCE, false>);
    case kLoopTP:
        return fastv ? reinterpret_cast<const void *>(&persistent_kernel<PRED, EXACT, kLoopTP, true>)
                     : reinterpret_cast<const void *>(&persistent_kernel<PRED, EXACT, kLoopTP, false>);
    default:
        return fastv ? reinterpret_cast<const void *>(&persistent_kernel<PRED, true, kLoopDO, true>)
                     : reinterpret_cast<const void *>(&persistent_kernel<PRED, true, kLoopDO, false>);
    }
}

// fastv: the instantiation whose fast path keeps the visited bitmap in LDS
const void *persistent_select(int loop, bool pred, bool exact, bool fastv)
{
    if (pred) return exact ? persistent_ptr<true, true>(loop, fastv) : persistent_ptr<true, false>(loop, fastv);
    return exact ? persistent_ptr<false, true>(loop, fastv) : persistent_ptr<false, false>(loop, fastv);
}

bool uses_fast_visited(const SearchArgs &s) { return s.fast_visited && s.nodes <= kFastVisitedWords * 32; }

template <bool PRED, bool EXACT, int PHASE>
hipError_t launch_phase(const GraphArgs &g, const SearchArgs &s, Cursor c, int grid, hipStream_t st, int *launches)
{
    if (PHASE == kPhaseContract && s.slabs && !s.tile_status) {
        const int marking = std::min(grid, s.slab_count);
        hipLaunchKernelGGL((contract_bits_kernel<PRED, EXACT>), dim3(marking), dim3(kBlock), 0, st, g, s, c);
        hipLaunchKernelGGL((contract_collect_kernel<EXACT>), dim3(marking), dim3(kBlock), 0, st, g, s, c);
        *launches += 2;
        return hipGetLastError();
    }
    hipLaunchKernelGGL((step_kernel<PRED, EXACT, PHASE>), dim3(grid), dim3(kBlock), 0, st, g, s, c);
    (*launches)++;
    if (PHASE == kPhaseExpandContract || PHASE == kPhaseContractExpand || PHASE == kPhaseExpand) {
        hipLaunchKernelGGL((hub_kernel<PRED, EXACT, PHASE>), dim3(grid), dim3(kBlock), 0, st, g, s, c);
        (*launches)++;
    }
    return hipGetLastError();
}

template <bool PRED, bool EXACT>
hipError_t launch_step_t(int phase, const GraphArgs &g, const SearchArgs &s, Cursor c, int grid, hipStream_t st,
                         int *launches)
{
    switch (phase) {
    case kPhaseExpandContract: return launch_phase<PRED, true, kPhaseExpandContract>(g, s, c, grid, st, launches);
    case kPhaseContractExpand: return launch_phase<PRED, EXACT, kPhaseContractExpand>(g, s, c, grid, st, launches);
    case kPhaseContract: return launch_phase<PRED, EXACT, kPhaseContract>(g, s, c, grid, st, launches);
    case kPhaseExpand: return launch_phase<PRED, EXACT, kPhaseExpand>(g, s, c, grid, st, launches);
    case kPhaseFilter: return launch_phase<PRED, EXACT, kPhaseFilter>(g, s, c, grid, st, launches);
    case kPhaseBottomUp: return launch_phase<PRED, true, kPhaseBottomUp>(g, s, c, grid, st, launches);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

int adjacency_width(int nodes, int max_degree)
{
    if (nodes > kFastVisitedWords * 32 || max_degree < 1 || max_degree > kAdjMaxDegree) return 0;
    return max_degree <= 4 ? 4 : 8;
}

hipError_t launch_adjacency(const int *row, const int *col, int nodes, int width, unsigned *adj, hipStream_t st)
{
    const long long count = (long long) nodes * width;
    const int grid = (int) std::min<long long>(16384, (count + 255) / 256);
    hipLaunchKernelGGL(adjacency_kernel, dim3(grid), dim3(256), 0, st, row, col, nodes, width, adj);
    return hipGetLastError();
}

hipError_t launch_reset_labels(int *depth, int *pred, unsigned *visited, int nodes, hipStream_t st)
{
    int grid = (nodes + 255) / 256;
    if (grid > 16384) grid = 16384;
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL(reset_labels_kernel, dim3(grid), dim3(256), 0, st, depth, pred, visited, nodes);
    return hipGetLastError();
}

hipError_t launch_init_search(const SearchArgs &s, const int *row, int src, int label_source, bool reset,
                              hipStream_t st)
{
    int grid = 1;
    if (reset) grid = std::min(16384, std::max(1, (s.nodes + 255) / 256));
    hipLaunchKernelGGL(init_search_kernel, dim3(grid), dim3(256), 0, st, s, row, src, label_source, reset ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_queue_from_bitmap(const SearchArgs &s, Cursor c, int grid, hipStream_t st, int *launches)
{
    GraphArgs g{nullptr, nullptr, s.nodes, nullptr, nullptr};
    hipLaunchKernelGGL(queue_from_bitmap_kernel, dim3(grid), dim3(kBlock), 0, st, g, s, c);
    (*launches)++;
    return hipGetLastError();
}

hipError_t launch_build_frontier_bitmap(const SearchArgs &s, Cursor c, int grid, hipStream_t st, int *launches)
{
    GraphArgs g{nullptr, nullptr, s.nodes, nullptr, nullptr};
    for (int pass = 0; pass < 2; pass++) {
        hipLaunchKernelGGL(frontier_bitmap_kernel, dim3(grid), dim3(kBlock), 0, st, g, s, c, pass);
        (*launches)++;
    }
    return hipGetLastError();
}

hipError_t launch_step(int phase, bool pred, bool exact, const GraphArgs &g, const SearchArgs &s, Cursor c,
                       int grid, hipStream_t st, int *launches)
{
    if (pred) return exact ? launch_step_t<true, true>(phase, g, s, c, grid, st, launches)
                           : launch_step_t<true, false>(phase, g, s, c, grid, st, launches);
    return exact ? launch_step_t<false, true>(phase, g, s, c, grid, st, launches)
                 : launch_step_t<false, false>(phase, g, s, c, grid, st, launches);
}

hipError_t launch_coresident(const void *kernel, dim3 grid, dim3 block, void **args, hipStream_t st)
{
    static std::atomic<bool> plain{false};
    if (!plain.load(std::memory_order_relaxed)) {
        hipError_t e = hipLaunchCooperativeKernel(kernel, grid, block, args, 0, st);
        if (e != hipErrorIllegalState) return e;
        (void) hipGetLastError();  // the refusal is not an error of this launch
        plain.store(true, std::memory_order_relaxed);
    }
    return hipLaunchKernel(kernel, grid, block, args, 0, st);
}

hipError_t launch_persistent(int loop, bool pred, bool exact, const GraphArgs &g, const SearchArgs &s, Cursor c,
                             int grid, hipStream_t st)
{
    GraphArgs ga = g;
    SearchArgs sa = s;
    Cursor ca = c;
    void *args[] = {&ga, &sa, &ca};
    return launch_coresident(persistent_select(loop, pred, exact, uses_fast_visited(s)), dim3(grid), dim3(kBlock),
                             args, st);
}

// The smaller of the two instantiations' occupancies (which one a search
// launches depends on the graph and the configuration).
int persistent_max_blocks_per_cu(int loop, bool pred, bool exact)
{
    int blocks = 1 << 30;
    for (int fastv = 0; fastv < 2; fastv++) {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, persistent_select(loop, pred, exact, fastv != 0), kBlock,
                                                         0) != hipSuccess)
            return 0;
        blocks = std::min(blocks, b);
    }
    return blocks;
}

int step_max_blocks_per_cu(bool pred)
{
    int blocks = 0;
    const void *k = pred ? reinterpret_cast<const void *>(&step_kernel<true, true, kPhaseExpandContract>)
                         : reinterpret_cast<const void *>(&step_kernel<false, true, kPhaseExpandContract>);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, kBlock, 0) != hipSuccess) return 0;
    return blocks;
}

int barrier_bench_max_blocks_per_cu()
{
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void *>(&barrier_bench_kernel),
                                                     kBlock, 0) != hipSuccess)
        return 0;
    return blocks;
}

hipError_t launch_barrier_bench(Control *ctl, int iterations, int grid, hipStream_t st)
{
    Control *c = ctl;
    int it = iterations;
    void *args[] = {&c, &it};
    return launch_coresident(reinterpret_cast<const void *>(&barrier_bench_kernel), dim3(grid), dim3(kBlock), args,
                             st);
}

hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t st)
{
    size_t n = bytes / 16;
    hipLaunchKernelGGL(b40c_calibration_copy_kernel, dim3(2048), dim3(256), 0, st,
                       reinterpret_cast<const uint4 *>(src), reinterpret_cast<uint4 *>(dst), n);
    return hipGetLastError();
}

hipError_t launch_wave_selftest(const int *in, int *out_scan, int *out_rank, int n, hipStream_t st)
{
    int grid = (n + kWave - 1) / kWave;
    hipLaunchKernelGGL(wave_selftest_kernel, dim3(grid), dim3(kWave), 0, st, in, out_scan, out_rank, n);
    return hipGetLastError();
}

}  // namespace b40c_hip
