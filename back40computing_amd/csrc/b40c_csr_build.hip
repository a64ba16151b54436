// b40c_csr_build.hip -- CSR construction on the device (C ABI in
// include/b40c_graph.h, b40c_device_csr_*).
//
// The reference builds every CSR on the host: CsrGraph::FromCoo stable-sorts
// the COO tuples by row (b40c/graph/csr_graph.cuh:108-152), after builders
// and file readers produced them (b40c/graph/builder/*.cuh).  Here the
// tuples become 64-bit keys (row << b | column, b = bits of V - 1) that an
// LSD radix sort orders on the device (digits of up to 9 bits, 2b bits in all: a
// per-tile digit histogram, one chained scan of the digit-major count matrix,
// then a stable scatter ranked by wave ballots); duplicates are dropped by a
// chained stream compaction; row offsets are written at the row boundaries
// of the sorted keys.  Rows come out sorted by column, as the host builder
// (graph_builder.cpp) makes them, so the two agree bit for bit.
//
// Self-loops to drop become the key of (2^b - 1, 2^b - 1), itself a loop, so
// they sort after every kept key and are cut off by count.
#include "b40c_graph.h"
#include "b40c_primitives.hpp"
#include "b40c_scan_internal.hpp"
#include "bfs_internal.hpp"
#include "graph_builder_internal.hpp"

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

using namespace b40c_hip;

namespace b40c_hip {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / prim::kWave;
constexpr int kRounds = 16;                          // keys per lane
constexpr int kTile = kThreads * kRounds;            // 4096 keys per tile
constexpr int kWaveKeys = prim::kWave * kRounds;     // 1024 contiguous keys per wave
constexpr int kDigitBits = 9;                        // most bits per sorting pass
constexpr int kDigits = 1 << kDigitBits;

__device__ __forceinline__ unsigned digit_of(unsigned long long key, int shift, int bits)
{
    return (unsigned) (key >> shift) & ((1u << bits) - 1u);
}

// Per-tile digit counts, digit-major: counts[d * tiles + tile].
__global__ __launch_bounds__(kThreads) void sort_upsweep_kernel(const unsigned long long *keys, long long n, int shift,
                                                                int bits, unsigned *counts, long long tiles)
{
    __shared__ unsigned hist[kDigits];
    const int digits = 1 << bits;
    for (int d = threadIdx.x; d < digits; d += kThreads) hist[d] = 0u;
    __syncthreads();
    const long long tile = blockIdx.x;
    const int wave = threadIdx.x / prim::kWave, lane = prim::lane();
    const long long base = tile * kTile + (long long) wave * kWaveKeys + lane;
    unsigned long long key[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const long long i = base + (long long) r * prim::kWave;
        key[r] = i < n ? keys[i] : 0ull;
    }
#pragma unroll
    for (int r = 0; r < kRounds; r++)
        if (base + (long long) r * prim::kWave < n) atomicAdd(&hist[digit_of(key[r], shift, bits)], 1u);
    __syncthreads();
    for (int d = threadIdx.x; d < digits; d += kThreads) counts[(long long) d * tiles + tile] = hist[d];
}

// Stable scatter by digit.  Wave w of a tile owns keys [w * 1024, (w + 1) *
// 1024) of the tile and walks them in 16 rounds of 64; a key's slot is its
// digit's scanned offset for this tile, plus the keys of that digit in the
// tile's lower waves, plus those earlier in its own wave (ballot match of
// the digit bits).
__global__ __launch_bounds__(kThreads) void sort_downsweep_kernel(const unsigned long long *keys_in,
                                                                  unsigned long long *keys_out, long long n, int shift,
                                                                  int bits, const unsigned *offsets, long long tiles)
{
    __shared__ unsigned base_of[kWaves][kDigits];
    const int digits = 1 << bits;
    for (int d = threadIdx.x; d < digits; d += kThreads)
        for (int w = 0; w < kWaves; w++) base_of[w][d] = 0u;
    __syncthreads();
    const long long tile = blockIdx.x;
    const int wave = threadIdx.x / prim::kWave, lane = prim::lane();
    const long long base = tile * kTile + (long long) wave * kWaveKeys + lane;
    unsigned long long key[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const long long i = base + (long long) r * prim::kWave;
        key[r] = i < n ? keys_in[i] : 0ull;
    }
#pragma unroll
    for (int r = 0; r < kRounds; r++)
        if (base + (long long) r * prim::kWave < n) atomicAdd(&base_of[wave][digit_of(key[r], shift, bits)], 1u);
    __syncthreads();
    for (int d = threadIdx.x; d < digits; d += kThreads) {
        // this tile's offset, then the lower waves' counts
        unsigned run = offsets[(long long) d * tiles + tile];
        for (int w = 0; w < kWaves; w++) {
            const unsigned c = base_of[w][d];
            base_of[w][d] = run;
            run += c;
        }
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const long long i = base + (long long) r * prim::kWave;
        const bool valid = i < n;
        const unsigned d = digit_of(key[r], shift, bits);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kDigitBits; b++) {  // (bits past the digit's are clear in all)
            const bool bit = (d >> b) & 1u;
            const uint64_t m = __ballot(valid && bit);
            peers &= bit ? m : ~m;
        }
        // every lane reads its digit's base before the group's first lane
        // advances it (one wave's LDS operations complete in order)
        const unsigned at = base_of[wave][d];
        const int rank = __popcll(peers & below);
        if (valid) {
            keys_out[at + (unsigned) rank] = key[r];
            if (rank == 0) base_of[wave][d] = at + (unsigned) __popcll(peers);
        }
    }
}

// What a keys kernel counts; read back before the sort.
struct KeyCounts {
    unsigned long long loops;  // keys dropped
    unsigned outside;          // pairs with an end outside the graph
    unsigned pad;
};

// Keys of (src, dst) pairs; with symmetrize also (dst, src); self-loops to
// drop become the loop key (2^b - 1, 2^b - 1) and are counted.  Pairs with
// an end outside [0, nodes) are counted too (the caller rejects the list).
__global__ __launch_bounds__(kThreads) void pair_keys_kernel(const int *src, const int *dst, long long pairs, int nodes,
                                                             int bits, int symmetrize, int drop_loops,
                                                             unsigned long long *keys, KeyCounts *counts)
{
    unsigned outside = 0;
    const unsigned long long loop_key = ((1ull << bits) - 1ull) << bits | ((1ull << bits) - 1ull);
    unsigned long long dropped = 0;
    for (long long i = blockIdx.x * (long long) kThreads + threadIdx.x; i < pairs;
         i += (long long) gridDim.x * kThreads) {
        const unsigned long long u = (unsigned) src[i], v = (unsigned) dst[i];
        if (u >= (unsigned) nodes || v >= (unsigned) nodes) outside++;
        const bool drop = drop_loops && u == v;
        const long long at = symmetrize ? 2 * i : i;
        keys[at] = drop ? loop_key : (u << bits) | v;
        if (symmetrize) keys[at + 1] = drop ? loop_key : (v << bits) | u;
        if (drop) dropped += symmetrize ? 2 : 1;
    }
    if (dropped) atomicAdd(&counts->loops, dropped);
    if (outside) atomicAdd(&counts->outside, outside);
}

// SplitMix64 (Steele, Lea, Flood, OOPSLA 2014) and the counter-based stream of
// the host builders (graph_builder.cpp), so device samples equal host ones.
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

constexpr unsigned long long kGolden = 0x9E3779B97F4A7C15ull;

// Graph500-style R-MAT samples (one per e), scrambled through perm, emitted
// as symmetric keys with loops dropped, exactly as b40c_graph_rmat draws them.
__global__ __launch_bounds__(kThreads) void rmat_keys_kernel(long long samples, int scale, unsigned long long seed,
                                                             unsigned long long t_a, unsigned long long t_ab,
                                                             unsigned long long t_abc, const int *perm, int bits,
                                                             unsigned long long *keys, unsigned long long *loops)
{
    const unsigned long long loop_key = ((1ull << bits) - 1ull) << bits | ((1ull << bits) - 1ull);
    unsigned long long dropped = 0;
    for (long long e = blockIdx.x * (long long) kThreads + threadIdx.x; e < samples;
         e += (long long) gridDim.x * kThreads) {
        unsigned long long s = mix64(seed ^ mix64((unsigned long long) e * kGolden + 0x632BE59BD9B4E019ull));
        unsigned u = 0, v = 0;
        unsigned long long draw = 0;
        for (int lvl = 0; lvl < scale; lvl++) {
            if ((lvl & 1) == 0) {
                s += kGolden;
                draw = mix64(s);
            }
            const unsigned long long r = (lvl & 1) ? (draw >> 32) : (draw & 0xFFFFFFFFull);
            unsigned ub, vb;
            if (r < t_a) { ub = 0; vb = 0; }
            else if (r < t_ab) { ub = 0; vb = 1; }
            else if (r < t_abc) { ub = 1; vb = 0; }
            else { ub = 1; vb = 1; }
            u = (u << 1) | ub;
            v = (v << 1) | vb;
        }
        if (perm) {
            u = (unsigned) perm[u];
            v = (unsigned) perm[v];
        }
        const bool drop = u == v;
        keys[2 * e] = drop ? loop_key : ((unsigned long long) u << bits) | v;
        keys[2 * e + 1] = drop ? loop_key : ((unsigned long long) v << bits) | u;
        if (drop) dropped += 2;
    }
    if (dropped) atomicAdd(loops, dropped);
}

// Chained stable compaction of sorted keys: keeps key i when it differs from
// key i - 1 (consecutive duplicates collapse to the first).  Wave w of a tile
// owns 1024 consecutive keys and walks them in rounds of 64, so every load
// and store instruction covers consecutive keys (sixteen consecutive keys a
// thread made 8 M keys 100 us; 49 us now).
__global__ __launch_bounds__(kThreads) void unique_kernel(const unsigned long long *in, unsigned long long *out,
                                                          long long n, ChainArgs c, unsigned *d_count)
{
    __shared__ long long s_tile;
    __shared__ unsigned s_wave[kWaves], s_prefix;
    const long long tile = prim::take_tile(c, &s_tile);
    const int wave = threadIdx.x / prim::kWave, lane = prim::lane();
    const long long base = tile * kTile + (long long) wave * kWaveKeys;
    unsigned long long v[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const long long i = base + r * prim::kWave + lane;
        v[r] = i < n ? in[i] : 0ull;
    }
    unsigned long long before = base > 0 && base <= n ? in[base - 1] : 0ull;  // the key before the round's first
    uint64_t keep[kRounds];
    unsigned run = 0;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const long long i = base + r * prim::kWave + lane;
        unsigned long long prev = __shfl_up(v[r], 1);
        if (lane == 0) prev = before;
        keep[r] = __ballot(i < n && (i == 0 || v[r] != prev));
        run += (unsigned) __popcll(keep[r]);
        before = __shfl(v[r], prim::kWave - 1);
    }
    if (lane == 0) s_wave[wave] = run;
    __syncthreads();
    unsigned off = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        if (w < wave) off += s_wave[w];
        agg += s_wave[w];
    }
    const unsigned prefix = prim::chain_prefix(c, tile, agg, &s_prefix);
    unsigned at = prefix + off;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        if ((keep[r] >> lane) & 1u) out[at + (unsigned) prim::lanes_below(keep[r])] = v[r];
        at += (unsigned) __popcll(keep[r]);
    }
    if (tile == c.tiles - 1 && threadIdx.x == 0) *d_count = prefix + agg;
}

// Columns and row offsets from E sorted keys: key i starts row u = key >> b,
// and writes row[w] = i for every w in (row of key i - 1, u]; the last key
// closes the rows after it with E.
__global__ __launch_bounds__(kThreads) void csr_from_keys_kernel(const unsigned long long *keys, long long edges,
                                                                 int bits, int nodes, int *row, int *col)
{
    const unsigned long long mask = (1ull << bits) - 1ull;
    for (long long i = blockIdx.x * (long long) kThreads + threadIdx.x; i < edges;
         i += (long long) gridDim.x * kThreads) {
        const unsigned long long k = keys[i];
        const int u = (int) (k >> bits);
        col[i] = (int) (k & mask);
        const int prev = i == 0 ? -1 : (int) (keys[i - 1] >> bits);
        for (int w = prev + 1; w <= u; w++) row[w] = (int) i;
        if (i == edges - 1)
            for (int w = u + 1; w <= nodes; w++) row[w] = (int) edges;
    }
}

__global__ __launch_bounds__(kThreads) void fill_int_kernel(int *p, long long n, int value)
{
    for (long long i = blockIdx.x * (long long) kThreads + threadIdx.x; i < n; i += (long long) gridDim.x * kThreads)
        p[i] = value;
}

// Last u in [0, nodes) with row[u] <= e.
__device__ __forceinline__ int row_of_edge(const int *row, int nodes, long long e)
{
    int lo = 0, hi = nodes - 1;
    while (lo < hi) {
        const int mid = lo + (hi - lo + 1) / 2;
        if ((long long) row[mid] <= e) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// (column, row) keys of every edge of a CSR: the transpose's tuples.  A tile
// of 4096 edges finds its first and last row by two searches; the rows
// starting inside it leave their numbers at their first edges in LDS (the
// last of several starting at one edge is the one with edges), and a running
// maximum hands every edge its row.  (A search per edge, 20 dependent loads,
// made 16 M edges 249 us; 55 now.)
// A tile of more than kWalkRows rows an edge searches all the same, a thread's
// edges kSearches at a time (sixteen at a time took 104 registers and half the
// waves from the tiles that walk: 16 M edges 85 us instead of 54): its empty
// rows have no bound, and one workgroup walked all of them (whole transposes
// of 1000 edges over 2^21 vertices 3051 us walked, 690 searched; of 5000 over
// 20 M 19360 and 1310; 300 k over 2^21, seven rows an edge, 90 either way).
constexpr int kWalkRows = 4;
constexpr int kSearches = 4;

__global__ __launch_bounds__(kThreads) void transpose_keys_kernel(const int *row, const int *col, int nodes,
                                                                  long long edges, int bits,
                                                                  unsigned long long *keys)
{
    __shared__ int s_row[kTile];
    __shared__ int s_wave[kWaves], s_first, s_last;
    const long long e0 = (long long) blockIdx.x * kTile;
    const int count = (int) (edges - e0 < (long long) kTile ? edges - e0 : (long long) kTile);
    for (int i = threadIdx.x; i < kTile; i += kThreads) s_row[i] = 0;
    if (threadIdx.x == 0) s_first = row_of_edge(row, nodes, e0);
    if (threadIdx.x == prim::kWave) s_last = row_of_edge(row, nodes, e0 + count - 1);
    __syncthreads();
    const int first = s_first, last = s_last;
    if (last - first > kWalkRows * kTile) {  // workgroup-uniform
        int top = 1;  // (last - first < 2^31)
        while (top <= (last - first) / 2) top *= 2;
#pragma unroll 1
        for (int k0 = 0; k0 * kThreads < count; k0 += kSearches) {
            int r[kSearches], e[kSearches];
#pragma unroll
            for (int k = 0; k < kSearches; k++) {
                r[k] = first;
                e[k] = (int) e0 + min((k0 + k) * kThreads + (int) threadIdx.x, count - 1);
            }
            for (int st = top; st > 0; st >>= 1) {
                int at[kSearches];
#pragma unroll
                for (int k = 0; k < kSearches; k++) at[k] = row[r[k] + min(st, last - r[k])];
#pragma unroll
                for (int k = 0; k < kSearches; k++)
                    if (st <= last - r[k] && at[k] <= e[k]) r[k] += st;
            }
#pragma unroll
            for (int k = 0; k < kSearches; k++) {
                const int i = (k0 + k) * kThreads + (int) threadIdx.x;
                if (i < count) keys[e0 + i] = ((unsigned long long) (unsigned) col[e0 + i] << bits) | (unsigned) r[k];
            }
        }
        return;
    }
    for (int u = first + 1 + (int) threadIdx.x; u <= last; u += kThreads) {
        const int at = (int) ((long long) row[u] - e0);
        if (at >= 0 && at < count) atomicMax(&s_row[at], u);
    }
    __syncthreads();
    // running maximum: sixteen consecutive edges a thread, then the threads before it
    int r[kRounds], top = 0;
#pragma unroll
    for (int k = 0; k < kRounds; k++) {
        top = max(top, s_row[threadIdx.x * kRounds + k]);
        r[k] = top;
    }
    int incl = top;
#pragma unroll
    for (int d = 1; d < prim::kWave; d <<= 1) {
        const int below = __shfl_up(incl, d);
        if (prim::lane() >= d) incl = max(incl, below);
    }
    const int wave = threadIdx.x / prim::kWave;
    if (prim::lane() == prim::kWave - 1) s_wave[wave] = incl;
    int before = __shfl_up(incl, 1);
    if (prim::lane() == 0) before = 0;
    __syncthreads();
    before = max(before, first);
    for (int w = 0; w < wave; w++) before = max(before, s_wave[w]);
#pragma unroll
    for (int k = 0; k < kRounds; k++) s_row[threadIdx.x * kRounds + k] = max(r[k], before);
    __syncthreads();
    for (int i = threadIdx.x; i < count; i += kThreads)
        keys[e0 + i] = ((unsigned long long) (unsigned) col[e0 + i] << bits) | (unsigned) s_row[i];
}

unsigned grid_for(long long n)
{
    return (unsigned) std::max(1LL, std::min((n + kThreads - 1) / kThreads, 16384LL));
}

int bits_for(int nodes)
{
    int b = 1;
    while (b < 31 && (1LL << b) < (long long) nodes) b++;
    return b;
}

// What a build needs besides its result -- a stream, events, chain state and
// its buffers -- is kept per device between builds: allocating and freeing 260
// MB took longer than transposing 16 M edges (1.3 ms of 2.7, on some boxes 8
// of 9.5).  One build at a time has the kept set; others at the same time make
// their own.  The buffers stay below kKeepBytes in all, and go back to the
// device when the last device CSR built here is freed, or when an allocation
// of the library finds no room (device_malloc, run_build).  They are separate
// allocations: the runtime hands small ones that were freed out again at once,
// where one block of all of them left it to map new memory for the problem
// that is usually made next (R-MAT scale 13: 765 instead of 470 us).
constexpr size_t kKeepBytes = (size_t) 512 << 20;
constexpr int kKeepDevices = 64;

// (the keys twice, the digit counts, the vertex permutation, the pairs)
enum Buffer { kKeys0, kKeys1, kCounts, kPerm, kSrc, kDst, kBuffers };

struct BuildSet {
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    ChainState chain;
    void *buffer[kBuffers] = {};
    size_t bytes[kBuffers] = {};
    bool busy = false;

    hipError_t make(int device)
    {
        if (stream) return hipSuccess;
        hipError_t e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreate(&ev0);
        if (e == hipSuccess) e = hipEventCreate(&ev1);
        if (e == hipSuccess) e = chain.init(device);
        if (e != hipSuccess) drop();
        return e;
    }
    size_t held() const
    {
        size_t sum = 0;
        for (size_t b : bytes) sum += b;
        return sum;
    }
    hipError_t reserve(int k, size_t need)
    {
        if (need <= bytes[k]) return hipSuccess;
        release(k);
        hipError_t e = device_malloc(&buffer[k], need);
        if (e != hipSuccess) {
            buffer[k] = nullptr;
            return e;
        }
        bytes[k] = need;
        return hipSuccess;
    }
    void release(int k)
    {
        if (buffer[k]) (void) hipFree(buffer[k]);
        buffer[k] = nullptr;
        bytes[k] = 0;
    }
    void release_all()
    {
        for (int k = 0; k < kBuffers; k++) release(k);
    }
    void drop()
    {
        if (stream) (void) hipStreamSynchronize(stream);
        release_all();
        chain.release();
        if (ev0) (void) hipEventDestroy(ev0);
        if (ev1) (void) hipEventDestroy(ev1);
        if (stream) (void) hipStreamDestroy(stream);
        ev0 = ev1 = nullptr;
        stream = nullptr;
    }
};

std::mutex g_keep_mu;
BuildSet g_keep[kKeepDevices];
int64_t g_live[kKeepDevices];  // device CSRs built and not yet freed

// One build: the kept set of its device, or a set of its own.
struct Builder {
    int device = 0;
    BuildSet own, *set = nullptr;
    hipStream_t stream = nullptr;
    unsigned long long *keys[2] = {nullptr, nullptr};
    unsigned *counts = nullptr;
    int *perm = nullptr;
    int *src = nullptr, *dst = nullptr;
    int status = 0;  // first failure: 1 invalid, 2 out of memory, 4 device error
    size_t need = 0; // bytes of buffers that the build uses

    ~Builder()
    {
        if (!set) return;
        if (stream) (void) hipStreamSynchronize(stream);
        if (set == &own) {
            own.drop();
            return;
        }
        std::lock_guard<std::mutex> lock(g_keep_mu);
        if (set->held() > kKeepBytes || g_live[device] == 0) set->release_all();
        set->busy = false;
    }

    // After a build that ran out of memory: whether the kept buffers held more
    // than it needed; they are released.
    bool gives_room()
    {
        if (!set || set == &own || set->held() <= need) return false;
        (void) hipStreamSynchronize(stream);
        set->release_all();
        (void) hipGetLastError();
        return true;
    }

    bool ok(hipError_t e)
    {
        if (e == hipSuccess) return true;
        if (!status) status = e == hipErrorOutOfMemory ? 2 : 4;
        return false;
    }

    bool start(int dev)
    {
        device = dev;
        if (!ok(hipSetDevice(dev))) return false;
        set = &own;
        if (dev < kKeepDevices) {
            std::lock_guard<std::mutex> lock(g_keep_mu);
            if (!g_keep[dev].busy) {
                set = &g_keep[dev];
                set->busy = true;
            }
        }
        if (!ok(set->make(dev))) return false;
        stream = set->stream;
        return ok(hipEventRecord(set->ev0, stream));
    }

    // Device memory of a build over n keys, with a vertex permutation (perm_n
    // entries) and pairs (pairs_n), either of which may be none.
    bool alloc(long long n, long long perm_n, long long pairs_n)
    {
        const size_t keys_n = (size_t) std::max(1LL, n), tiles = (keys_n + kTile - 1) / kTile;
        const size_t want[kBuffers] = {sizeof(unsigned long long) * keys_n, sizeof(unsigned long long) * keys_n,
                                       sizeof(unsigned) * tiles * kDigits, sizeof(int) * (size_t) perm_n,
                                       sizeof(int) * (size_t) pairs_n, sizeof(int) * (size_t) pairs_n};
        for (size_t w : want) need += w;
        for (int k = 0; k < kBuffers; k++)
            if (!ok(set->reserve(k, want[k]))) return false;
        keys[0] = static_cast<unsigned long long *>(set->buffer[kKeys0]);
        keys[1] = static_cast<unsigned long long *>(set->buffer[kKeys1]);
        counts = static_cast<unsigned *>(set->buffer[kCounts]);
        perm = static_cast<int *>(set->buffer[kPerm]);
        src = static_cast<int *>(set->buffer[kSrc]);
        dst = static_cast<int *>(set->buffer[kDst]);
        return true;
    }

    KeyCounts *key_counts() const { return reinterpret_cast<KeyCounts *>(set->chain.d_word); }

    bool read_key_counts(KeyCounts *c)
    {
        return ok(hipMemcpyAsync(c, key_counts(), sizeof(*c), hipMemcpyDeviceToHost, stream)) &&
               ok(hipStreamSynchronize(stream));
    }

    // LSD radix sort of keys[0][0, n) over bits [low_bit, key_bits); the result
    // is in keys[0].
    bool sort(long long n, int key_bits, int low_bit = 0)
    {
        if (n <= 1) return true;
        const long long tiles = (n + kTile - 1) / kTile;
        // as few passes as kDigitBits allow, then digits as narrow as those
        // passes allow: fewer digits leave longer runs per tile to write
        const int passes = std::max(1, (key_bits - low_bit + kDigitBits - 1) / kDigitBits);
        int cur = 0;
        for (int p = 0, shift = low_bit; p < passes; p++) {
            const int bits = (key_bits - shift + (passes - p) - 1) / (passes - p);
            const long long counts_n = tiles << bits;
            hipLaunchKernelGGL(sort_upsweep_kernel, dim3((unsigned) tiles), dim3(kThreads), 0, stream, keys[cur], n,
                               shift, bits, counts, tiles);
            if (!ok(hipGetLastError())) return false;
            ChainArgs c;
            if (!ok(set->chain.prepare(counts_n, scan_tile_items(counts_n), &c, stream))) return false;
            if (!ok(launch_scan_u32(counts, counts, counts_n, true, c, nullptr, stream))) return false;
            hipLaunchKernelGGL(sort_downsweep_kernel, dim3((unsigned) tiles), dim3(kThreads), 0, stream, keys[cur],
                               keys[cur ^ 1], n, shift, bits, counts, tiles);
            if (!ok(hipGetLastError())) return false;
            cur ^= 1;
            shift += bits;
        }
        if (cur == 1) std::swap(keys[0], keys[1]);
        return true;
    }

    // Number of kept keys after dropping `loops` trailing loop keys and, with
    // dedup, consecutive duplicates; the kept keys end up in keys[0].
    bool compact(long long n, long long loops, bool dedup, long long *kept)
    {
        long long m = n - loops;
        if (dedup && m > 0) {
            ChainArgs c;
            if (!ok(set->chain.prepare(m, kTile, &c, stream))) return false;
            hipLaunchKernelGGL(unique_kernel, dim3((unsigned) c.tiles), dim3(kThreads), 0, stream, keys[0], keys[1],
                               m, c, set->chain.d_word);
            if (!ok(hipGetLastError())) return false;
            unsigned k = 0;
            if (!ok(hipMemcpyAsync(&k, set->chain.d_word, sizeof(unsigned), hipMemcpyDeviceToHost, stream)) ||
                !ok(hipStreamSynchronize(stream)))
                return false;
            m = k;
            std::swap(keys[0], keys[1]);
        }
        *kept = m;
        return true;
    }

    bool finish(int nodes, long long edges, int bits, bool symmetric, b40c_device_csr *out)
    {
        if (edges > INT32_MAX) {
            if (!status) status = 3;
            return false;
        }
        int *row = nullptr, *col = nullptr;
        if (!ok(device_malloc(&row, sizeof(int) * ((size_t) nodes + 1))) ||
            !ok(device_malloc(&col, sizeof(int) * (size_t) std::max(1LL, edges)))) {
            if (row) (void) hipFree(row);
            return false;
        }
        if (edges == 0) hipLaunchKernelGGL(fill_int_kernel, dim3(grid_for(nodes + 1)), dim3(kThreads), 0, stream, row,
                                           (long long) nodes + 1, 0);
        else hipLaunchKernelGGL(csr_from_keys_kernel, dim3(grid_for(edges)), dim3(kThreads), 0, stream, keys[0],
                                edges, bits, nodes, row, col);
        float ms = 0.f;
        if (!ok(hipGetLastError()) || !ok(hipEventRecord(set->ev1, stream)) || !ok(hipEventSynchronize(set->ev1)) ||
            !ok(hipEventElapsedTime(&ms, set->ev0, set->ev1))) {
            (void) hipFree(row);
            (void) hipFree(col);
            return false;
        }
        out->device = device;
        out->nodes = nodes;
        out->edges = edges;
        out->row_offsets = row;
        out->column_indices = col;
        out->symmetric = symmetric ? 1 : 0;
        out->build_ms = ms;
        if (device < kKeepDevices) {
            std::lock_guard<std::mutex> lock(g_keep_mu);
            g_live[device]++;
        }
        return true;
    }
};

// Runs one build, and once more if it ran out of memory beside kept buffers
// larger than its own.
template <typename Build>
int run_build(int device, Build &&build)
{
    for (bool again = false;; again = true) {
        Builder b;
        const int rc = b.start(device) ? build(b) : b.status;
        if (rc != 2 || again || !b.gives_room()) return rc;
    }
}

int device_ok(int32_t device)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return 4;
    return device >= 0 && device < count ? 0 : 1;
}

bool pairs_inside(const int32_t *src, const int32_t *dst, int64_t pairs, int32_t nodes)
{
    for (int64_t i = 0; i < pairs; i++)
        if (src[i] < 0 || src[i] >= nodes || dst[i] < 0 || dst[i] >= nodes) return false;
    return true;
}

}  // namespace

hipError_t device_malloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    {
        std::lock_guard<std::mutex> lock(g_keep_mu);
        bool room = false;
        for (BuildSet &k : g_keep) {
            if (k.busy || !k.held()) continue;
            k.release_all();
            room = true;
        }
        if (!room) return e;
    }
    (void) hipGetLastError();
    return hipMalloc(p, bytes);
}

void device_csr_gone(int device)
{
    if (device < 0 || device >= kKeepDevices) return;
    std::lock_guard<std::mutex> lock(g_keep_mu);
    if (g_live[device] > 0 && --g_live[device] == 0 && !g_keep[device].busy) g_keep[device].release_all();
}

}  // namespace b40c_hip

extern "C" {

int b40c_device_csr_from_coo(int32_t device, int32_t nodes, int64_t num_pairs, const int32_t *h_src,
                             const int32_t *h_dst, int symmetrize, int dedup, int drop_self_loops,
                             b40c_device_csr *out)
{
    if (!out || nodes <= 0 || num_pairs < 0 || (num_pairs > 0 && (!h_src || !h_dst))) return 1;
    *out = b40c_device_csr{};
    const long long n = (symmetrize ? 2 : 1) * (long long) num_pairs;
    // the device checks the pairs; where it does not get to see them, they
    // are checked here (an invalid pair is the first error reported)
    auto unseen = [&](int rc) { return pairs_inside(h_src, h_dst, num_pairs, nodes) ? rc : 1; };
    if (n > (long long) UINT32_MAX) return unseen(3);  // (sort offsets are 32-bit)
    if (int rc = device_ok(device)) return unseen(rc);
    bool seen = n == 0;
    const int rc = run_build(device, [&](Builder &b) {
        const int bits = bits_for(nodes);
        long long edges = 0;
        if (n > 0) {
            const size_t pb = sizeof(int) * (size_t) num_pairs;
            KeyCounts kc;
            if (!b.alloc(n, 0, num_pairs) ||
                !b.ok(hipMemcpyAsync(b.src, h_src, pb, hipMemcpyHostToDevice, b.stream)) ||
                !b.ok(hipMemcpyAsync(b.dst, h_dst, pb, hipMemcpyHostToDevice, b.stream)) ||
                !b.ok(hipMemsetAsync(b.key_counts(), 0, sizeof(KeyCounts), b.stream)))
                return b.status;
            hipLaunchKernelGGL(pair_keys_kernel, dim3(grid_for(num_pairs)), dim3(kThreads), 0, b.stream, b.src, b.dst,
                               (long long) num_pairs, nodes, bits, symmetrize ? 1 : 0, drop_self_loops ? 1 : 0,
                               b.keys[0], b.key_counts());
            if (!b.ok(hipGetLastError()) || !b.read_key_counts(&kc)) return b.status;
            seen = true;
            if (kc.outside) return 1;
            if (!b.sort(n, 2 * bits) || !b.compact(n, (long long) kc.loops, dedup != 0, &edges)) return b.status;
        }
        if (!b.finish(nodes, edges, bits, symmetrize != 0, out)) return b.status ? b.status : 4;
        return 0;
    });
    return rc && !seen ? unseen(rc) : rc;
}

int b40c_device_csr_rmat(int32_t device, int32_t scale, int32_t edge_factor, double a, double b, double c,
                         uint64_t seed, int scramble, b40c_device_csr *out)
{
    if (!out || scale < 1 || scale > 30 || edge_factor < 1) return 1;
    if (a < 0 || b < 0 || c < 0 || a + b + c > 1.0) return 1;
    *out = b40c_device_csr{};
    const int32_t nodes = (int32_t) (1u << scale);
    const long long samples = (long long) edge_factor << scale;
    if (2 * samples > (long long) INT32_MAX * 2) return 3;
    if (int rc = device_ok(device)) return rc;
    const uint64_t two32 = 1ull << 32;
    const uint64_t t_a = (uint64_t) (a * two32), t_ab = (uint64_t) ((a + b) * two32),
                   t_abc = (uint64_t) ((a + b + c) * two32);
    std::vector<int32_t> perm;
    if (scramble) b40c_rmat_permutation(scale, seed, &perm);
    return run_build(device, [&](Builder &bld) {
        const int bits = scale;
        const long long n = 2 * samples;
        KeyCounts kc;
        if (!bld.alloc(n, scramble ? nodes : 0, 0) ||
            !bld.ok(hipMemsetAsync(bld.key_counts(), 0, sizeof(KeyCounts), bld.stream)))
            return bld.status;
        if (scramble && !bld.ok(hipMemcpyAsync(bld.perm, perm.data(), sizeof(int) * (size_t) nodes,
                                               hipMemcpyHostToDevice, bld.stream)))
            return bld.status;
        hipLaunchKernelGGL(rmat_keys_kernel, dim3(grid_for(samples)), dim3(kThreads), 0, bld.stream, samples, scale,
                           (unsigned long long) seed, (unsigned long long) t_a, (unsigned long long) t_ab,
                           (unsigned long long) t_abc, scramble ? bld.perm : nullptr, bits, bld.keys[0],
                           &bld.key_counts()->loops);
        if (!bld.ok(hipGetLastError()) || !bld.read_key_counts(&kc)) return bld.status;
        long long edges = 0;
        if (!bld.sort(n, 2 * bits) || !bld.compact(n, (long long) kc.loops, true, &edges)) return bld.status;
        if (!bld.finish(nodes, edges, bits, true, out)) return bld.status ? bld.status : 4;
        return 0;
    });
}

int b40c_device_csr_transpose(const b40c_device_csr *g, b40c_device_csr *out)
{
    if (!g || !out || g->nodes <= 0 || g->edges < 0 || !g->row_offsets) return 1;
    *out = b40c_device_csr{};
    if (int rc = device_ok(g->device)) return rc;
    return run_build(g->device, [&](Builder &b) {
        const int bits = bits_for(g->nodes);
        const long long n = g->edges;
        if (n > 0) {
            if (!b.alloc(n, 0, 0)) return b.status;
            hipLaunchKernelGGL(transpose_keys_kernel, dim3((unsigned) ((n + kTile - 1) / kTile)), dim3(kThreads), 0,
                               b.stream, g->row_offsets, g->column_indices, g->nodes, n, bits, b.keys[0]);
            // the tuples come in row order, and the passes are stable: sorting by
            // the column leaves every column's rows in order
            if (!b.ok(hipGetLastError()) || !b.sort(n, 2 * bits, bits)) return b.status;
        }
        if (!b.finish(g->nodes, n, bits, g->symmetric != 0, out)) return b.status ? b.status : 4;
        return 0;
    });
}

int b40c_device_csr_to_host(const b40c_device_csr *g, b40c_csr *out)
{
    if (!g || !out || g->nodes <= 0 || g->edges < 0 || !g->row_offsets) return 1;
    if (hipSetDevice(g->device) != hipSuccess) return 4;
    out->nodes = g->nodes;
    out->edges = g->edges;
    out->row_offsets = (int32_t *) std::malloc(sizeof(int32_t) * ((size_t) g->nodes + 1));
    out->column_indices = (int32_t *) std::malloc(sizeof(int32_t) * (size_t) std::max<int64_t>(g->edges, 1));
    if (!out->row_offsets || !out->column_indices) {
        b40c_graph_free(out);
        return 2;
    }
    if (hipMemcpy(out->row_offsets, g->row_offsets, sizeof(int32_t) * ((size_t) g->nodes + 1),
                  hipMemcpyDeviceToHost) != hipSuccess ||
        (g->edges > 0 && hipMemcpy(out->column_indices, g->column_indices, sizeof(int32_t) * (size_t) g->edges,
                                   hipMemcpyDeviceToHost) != hipSuccess)) {
        b40c_graph_free(out);
        return 4;
    }
    return 0;
}

void b40c_device_csr_free(b40c_device_csr *g)
{
    if (!g) return;
    if (g->row_offsets || g->column_indices) (void) hipSetDevice(g->device);
    if (g->row_offsets) device_csr_gone(g->device);
    if (g->row_offsets) (void) hipFree(g->row_offsets);
    if (g->column_indices) (void) hipFree(g->column_indices);
    g->row_offsets = g->column_indices = nullptr;
    g->nodes = 0;
    g->edges = 0;
}

}  // extern "C"
