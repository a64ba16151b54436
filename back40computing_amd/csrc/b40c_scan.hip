// b40c_scan.hip -- single-pass prefix scan and stable stream compaction
// (C ABI in include/b40c_scan.h).
//
// One kernel per call.  A workgroup takes the next tile index from an atomic
// counter, reduces its items (4096 to 16384), publishes the aggregate, looks back over
// the predecessors' status words for its exclusive prefix
// (prim::lookback_prefix), publishes its inclusive prefix and writes its
// outputs.  This replaces the reference's upsweep / spine / downsweep passes
// (b40c/scan/enactor.cuh:426-454, b40c/copy_if/enactor.cuh:436-461) and their
// spine storage.
#include "b40c_scan.h"
#include "b40c_primitives.hpp"
#include "b40c_scan_internal.hpp"
#include "bfs_internal.hpp"

#include <algorithm>
#include <mutex>

using namespace b40c_hip;

namespace b40c_hip {

namespace {

constexpr int kThreads = kScanThreads;
constexpr int kWaves = kThreads / prim::kWave;

// Wave-striped arrangement of a tile: wave w owns 64 * ITEMS consecutive
// items and reads them in rounds of 256, lane l taking four consecutive
// items at 4 l.  Each 16-byte load instruction of a wave then covers one
// contiguous KiB (a blocked arrangement touched 64 lines per instruction),
// and the items keep their order as (round, lane, item).  `fill` past the end.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Tiles of a large input stream through memory once: non-temporal (2^26
// items 135.9 -> 127.7 us; small inputs keep the caches for their reader).
template <int ROUNDS>
__device__ __forceinline__ void load_striped(const uint32_t *in, long long n, long long base, bool vec, uint32_t fill,
                                             uint4 (&v)[ROUNDS])
{
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const long long i = base + r * 256;
        if (vec && i + 4 <= n) {
            if constexpr (ROUNDS > 2) {
                const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(in + i));
                v[r] = make_uint4(t.x, t.y, t.z, t.w);
            } else {
                v[r] = *reinterpret_cast<const uint4 *>(in + i);
            }
        } else {
            v[r].x = i < n ? in[i] : fill;
            v[r].y = i + 1 < n ? in[i + 1] : fill;
            v[r].z = i + 2 < n ? in[i + 2] : fill;
            v[r].w = i + 3 < n ? in[i + 3] : fill;
        }
    }
}

__device__ __forceinline__ bool selected(uint32_t key, int op, uint32_t comparand)
{
    switch (op) {
    case B40C_SELECT_LESS: return key < comparand;
    case B40C_SELECT_NOT_EQUAL: return key != comparand;
    default: return (int32_t) key >= 0;
    }
}

// Bound: HBM, eight bytes per item.  The tile counter is one address whose
// atomics serialise (about 15 ns each, so 16385 tiles of 4096 items alone
// cost 245 us on 2^26 items): large inputs take tiles of 16384 items
// (ROUNDS = 8), small ones tiles of 4096 (ROUNDS = 2), which spread a short
// input over more workgroups (see scan_tile_items).
template <int ROUNDS>
__global__ __launch_bounds__(kThreads) void scan_kernel(const uint32_t *in, uint32_t *out, long long n, int exclusive,
                                                        int vec, ChainArgs c, uint32_t *d_total)
{
    __shared__ long long s_tile;
    __shared__ unsigned s_wave[kWaves], s_prefix;
    const long long tile = prim::take_tile(c, &s_tile);
    const int lane = prim::lane(), wave = threadIdx.x / prim::kWave;
    const long long base = tile * (kThreads * 4LL * ROUNDS) + (long long) wave * (256 * ROUNDS) + 4 * lane;
    uint4 v[ROUNDS];
    load_striped<ROUNDS>(in, n, base, vec != 0, 0u, v);
    unsigned off[ROUNDS], run = 0;  // sum of the wave's items before the lane's four of each round
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const unsigned sum = v[r].x + v[r].y + v[r].z + v[r].w;
        const unsigned incl = prim::wave_inclusive_sum_u32(sum);
        off[r] = run + incl - sum;
        run += (unsigned) __builtin_amdgcn_readlane((int) incl, prim::kWave - 1);
    }
    if (lane == 0) s_wave[wave] = run;
    __syncthreads();
    unsigned before = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        const unsigned t = s_wave[w];
        if (w < wave) before += t;
        agg += t;
    }
    const unsigned prefix = prim::chain_prefix(c, tile, agg, &s_prefix);
    const unsigned shift = prefix + before;
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const long long i = base + r * 256;
        const unsigned x = shift + off[r];
        uint4 o;
        if (exclusive) {
            o.x = x;
            o.y = o.x + v[r].x;
            o.z = o.y + v[r].y;
            o.w = o.z + v[r].z;
        } else {
            o.x = x + v[r].x;
            o.y = o.x + v[r].y;
            o.z = o.y + v[r].z;
            o.w = o.z + v[r].w;
        }
        if (vec && i + 4 <= n) {
            if constexpr (ROUNDS > 2)
                __builtin_nontemporal_store(u32x4{o.x, o.y, o.z, o.w}, reinterpret_cast<u32x4 *>(out + i));
            else
                *reinterpret_cast<uint4 *>(out + i) = o;
        } else {
            if (i < n) out[i] = o.x;
            if (i + 1 < n) out[i + 1] = o.y;
            if (i + 2 < n) out[i + 2] = o.z;
            if (i + 3 < n) out[i + 3] = o.w;
        }
    }
    if (d_total && tile == c.tiles - 1 && threadIdx.x == 0) {
        *d_total = prefix + agg;
        __threadfence_system();  // (may be pinned host memory)
    }
}

// Kept items are staged in LDS at their rank in the tile and leave it as
// consecutive words per wave (one contiguous run a tile), whatever the
// share that is kept.  Bound: HBM.
template <int ROUNDS>
__global__ __launch_bounds__(kThreads) void copy_if_kernel(const uint32_t *in, uint32_t *out, long long n, int op,
                                                           uint32_t comparand, int vec, ChainArgs c,
                                                           uint32_t *d_count, uint32_t *h_count)
{
    constexpr int kTileItems = kThreads * 4 * ROUNDS;
    __shared__ long long s_tile;
    __shared__ unsigned s_wave[kWaves], s_prefix;
    __shared__ uint32_t stage[kTileItems];
    const long long tile = prim::take_tile(c, &s_tile);
    const int lane = prim::lane(), wave = threadIdx.x / prim::kWave;
    const long long base = tile * (long long) kTileItems + (long long) wave * (256 * ROUNDS) + 4 * lane;
    uint4 v[ROUNDS];
    load_striped<ROUNDS>(in, n, base, vec != 0, 0u, v);
    unsigned keep = 0, run = 0, off[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const long long i = base + r * 256;
        unsigned m = 0;
        if (i < n && selected(v[r].x, op, comparand)) m |= 1u;
        if (i + 1 < n && selected(v[r].y, op, comparand)) m |= 2u;
        if (i + 2 < n && selected(v[r].z, op, comparand)) m |= 4u;
        if (i + 3 < n && selected(v[r].w, op, comparand)) m |= 8u;
        keep |= m << (4 * r);
        const unsigned cnt = (unsigned) __popc(m);
        const unsigned incl = prim::wave_inclusive_sum_u32(cnt);
        off[r] = run + incl - cnt;
        run += (unsigned) __builtin_amdgcn_readlane((int) incl, prim::kWave - 1);
    }
    static_assert(4 * ROUNDS <= 32, "one keep bit per item");
    if (lane == 0) s_wave[wave] = run;
    __syncthreads();
    unsigned before = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        const unsigned t = s_wave[w];
        if (w < wave) before += t;
        agg += t;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        unsigned at = before + off[r];
        const unsigned m = keep >> (4 * r);
        if (m & 1u) stage[at++] = v[r].x;
        if (m & 2u) stage[at++] = v[r].y;
        if (m & 4u) stage[at++] = v[r].z;
        if (m & 8u) stage[at++] = v[r].w;
    }
    // (chain_prefix's workgroup barrier orders the staging before its reads)
    const unsigned prefix = prim::chain_prefix(c, tile, agg, &s_prefix);
    for (unsigned i = threadIdx.x; i < agg; i += kThreads) {
        if constexpr (ROUNDS > 2) __builtin_nontemporal_store(stage[i], out + prefix + i);
        else out[prefix + i] = stage[i];
    }
    if (tile == c.tiles - 1 && threadIdx.x == 0) {
        if (d_count) *d_count = prefix + agg;
        if (h_count) *h_count = prefix + agg;
        __threadfence_system();
    }
}

__global__ void fill_u32_kernel(uint32_t *p, long long n, uint32_t value)
{
    for (long long i = blockIdx.x * (long long) blockDim.x + threadIdx.x; i < n; i += (long long) gridDim.x * blockDim.x)
        p[i] = value;
}

}  // namespace

// Inputs past 2^20 items take 16384-item tiles (see scan_kernel): there the
// tile counter, not the workgroups in flight, sets the pace (2^22 items:
// 26.8 us in tiles of 4096, 14.4 in tiles of 16384; 2^20 items, which are
// 256 of the small tiles: 10.4 us either way).  2^26 items: 249 us in tiles
// of 4096 read in a blocked arrangement, 130 us now (4.1 TB/s; a copy of
// the same size reaches 5.1).
int scan_tile_items(long long n) { return n > (1LL << 20) ? 16384 : 4096; }

hipError_t launch_scan_u32(const uint32_t *in, uint32_t *out, long long n, bool exclusive, const ChainArgs &c,
                           uint32_t *d_total, hipStream_t st)
{
    const int vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (scan_tile_items(n) == 16384)
        hipLaunchKernelGGL(scan_kernel<8>, dim3((unsigned) c.tiles), dim3(kThreads), 0, st, in, out, n,
                           exclusive ? 1 : 0, vec, c, d_total);
    else
        hipLaunchKernelGGL(scan_kernel<2>, dim3((unsigned) c.tiles), dim3(kThreads), 0, st, in, out, n,
                           exclusive ? 1 : 0, vec, c, d_total);
    return hipGetLastError();
}

// (8192: a 16384-item stage takes 64 KiB of LDS and leaves two workgroups
// per CU, 2^26 items keeping nearly all 169 us instead of 160)
int copy_if_tile_items(long long n) { return n > (1LL << 20) ? 8192 : 4096; }

hipError_t launch_copy_if_u32(const uint32_t *in, uint32_t *out, long long n, int op, uint32_t comparand,
                              const ChainArgs &c, uint32_t *d_count, uint32_t *h_count, hipStream_t st)
{
    const int vec = (reinterpret_cast<uintptr_t>(in) & 15) == 0;
    if (copy_if_tile_items(n) == 8192)
        hipLaunchKernelGGL(copy_if_kernel<4>, dim3((unsigned) c.tiles), dim3(kThreads), 0, st, in, out, n, op,
                           comparand, vec, c, d_count, h_count);
    else
        hipLaunchKernelGGL(copy_if_kernel<2>, dim3((unsigned) c.tiles), dim3(kThreads), 0, st, in, out, n, op,
                           comparand, vec, c, d_count, h_count);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Allocation-free scan (b40c_scan_noalloc): the tile counter and the status
// words live in one file-scope device array per GPU.  Word 0 is the counter;
// the status words start at word kNoAllocStatus (a 256-byte line of their
// own).  Every call clears what it uses with a fill kernel (no memset node
// if the caller captures the call in a graph) and uses epoch 0.
// ---------------------------------------------------------------------------
namespace {

constexpr long long kNoAllocMaxItems = 1LL << 26;
constexpr long long kNoAllocMaxTiles = 16384;  // (of at least 4096 items)
constexpr int kNoAllocStatus = 32;
constexpr int kNoAllocDevices = 64;

static __device__ __align__(256) unsigned long long scratch[kNoAllocStatus + kNoAllocMaxTiles];

__global__ __launch_bounds__(kThreads) void noalloc_clear_kernel(unsigned long long *words, long long tiles)
{
    for (long long i = blockIdx.x * (long long) kThreads + threadIdx.x; i < tiles; i += (long long) gridDim.x * kThreads)
        words[kNoAllocStatus + i] = 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) words[0] = 0ull;
}

std::mutex g_noalloc_mu;
unsigned long long *g_noalloc_ptr[kNoAllocDevices];  // device address of `scratch`, per device

// The device address of this device's `scratch` (the array's name is a host
// stand-in, not a device address), looked up once per device.
hipError_t noalloc_scratch(int device, unsigned long long **out)
{
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[device]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_noalloc_ptr[device] = static_cast<unsigned long long *>(ptr);
    }
    *out = g_noalloc_ptr[device];
    return hipSuccess;
}

}  // namespace

// ---------------------------------------------------------------------------
// Pinned host words for enactors' totals, handed out from one page that the
// process keeps (pinning memory for every enactor took 55 us of its creation);
// past the page's words an enactor pins its own.
// ---------------------------------------------------------------------------
namespace {

constexpr int kPinnedWords = 1024;
std::mutex g_word_mu;
uint32_t *g_word_page = nullptr;
bool g_word_used[kPinnedWords];

hipError_t take_pinned_word(uint32_t **word)
{
    std::lock_guard<std::mutex> lock(g_word_mu);
    if (!g_word_page) {
        hipError_t e = hipHostMalloc(&g_word_page, kPinnedWords * sizeof(uint32_t), hipHostMallocPortable);
        if (e != hipSuccess) {
            g_word_page = nullptr;
            return e;
        }
    }
    for (int i = 0; i < kPinnedWords; i++) {
        if (g_word_used[i]) continue;
        g_word_used[i] = true;
        *word = g_word_page + i;
        return hipSuccess;
    }
    return hipHostMalloc(word, sizeof(uint32_t), hipHostMallocPortable);
}

void give_pinned_word(uint32_t *word)
{
    std::lock_guard<std::mutex> lock(g_word_mu);
    if (g_word_page && word >= g_word_page && word < g_word_page + kPinnedWords) g_word_used[word - g_word_page] = false;
    else (void) hipHostFree(word);
}

}  // namespace

// ---------------------------------------------------------------------------
// Chain state: the tile counter and the per-tile status words.
// ---------------------------------------------------------------------------
hipError_t ChainState::init(int dev)
{
    device = dev;
    hipError_t e = device_malloc(&d_counter, sizeof(unsigned long long) + 4 * sizeof(uint32_t));
    if (e != hipSuccess) return e;
    d_word = reinterpret_cast<uint32_t *>(d_counter + 1);
    return hipSuccess;
}

hipError_t ChainState::prepare(long long items, int tile_items, ChainArgs *c, hipStream_t st)
{
    if (epoch == 0) {
        // The first launch: its tile counter starts at zero.  Cleared on the
        // launches' own stream: non-blocking streams do not wait for the null
        // stream, whose fill may still run when hipMemset returns.
        hipError_t e = hipMemsetAsync(d_counter, 0, sizeof(unsigned long long), st);
        if (e != hipSuccess) return e;
    }
    const long long tiles = std::max(1LL, (items + tile_items - 1) / tile_items);
    if (tiles > capacity) {
        // earlier launches on the stream may still read the old words
        if (d_status) {
            hipError_t e = hipStreamSynchronize(st);
            if (e != hipSuccess) return e;
            (void) hipFree(d_status);
        }
        d_status = nullptr;
        capacity = 0;
        hipError_t e = device_malloc(&d_status, sizeof(unsigned long long) * (size_t) tiles);
        if (e != hipSuccess) return e;
        // state 0 (unpublished) under every epoch; ordered on the launch's
        // (non-blocking) stream
        if ((e = hipMemsetAsync(d_status, 0, sizeof(unsigned long long) * (size_t) tiles, st)) != hipSuccess)
            return e;
        capacity = tiles;
    }
    epoch = (epoch + 1) & 0x3FFFFFFFu;
    if (epoch == 0) {
        // the 30-bit epoch wrapped: older words could match again
        hipError_t e = hipMemsetAsync(d_status, 0, sizeof(unsigned long long) * (size_t) capacity, st);
        if (e != hipSuccess) return e;
        epoch = 1;
    }
    c->status = d_status;
    c->tile_counter = d_counter;
    c->epoch = epoch;
    c->tiles = tiles;
    return hipSuccess;
}

void ChainState::release()
{
    if (d_status) (void) hipFree(d_status);
    if (d_counter) (void) hipFree(d_counter);
    d_status = nullptr;
    d_counter = nullptr;
    capacity = 0;
}

}  // namespace b40c_hip

struct b40c_scan_enactor {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    ChainState chain;
    // Pinned host word the last tile of a launch writes its total to: the
    // host reads it once the launch's stop event has passed, with no copy
    // of its own (about 25 us of a call).
    uint32_t *h_word = nullptr, *h_word_dev = nullptr;
    float last_ms = 0.f;
};

namespace {

bfs_status timed_sync(b40c_scan_enactor *e)
{
    hipError_t r;
    if ((r = hipEventRecord(e->ev1, e->stream)) != hipSuccess) return host_hip_fail(r, "record");
    if ((r = hipEventSynchronize(e->ev1)) != hipSuccess) return host_hip_fail(r, "synchronize");
    if ((r = hipEventElapsedTime(&e->last_ms, e->ev0, e->ev1)) != hipSuccess) return host_hip_fail(r, "elapsed");
    return BFS_OK;
}

}  // namespace

extern "C" {

bfs_status b40c_scan_enactor_create(int32_t device, b40c_scan_enactor **out)
{
    if (!out) return host_fail(BFS_ERR_INVALID_ARG, "null output handle");
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return host_fail(BFS_ERR_NO_DEVICE, "no HIP device");
    if (device < 0 || device >= count) return host_fail(BFS_ERR_INVALID_ARG, "device ordinal out of range");
    hipError_t e;
    if ((e = hipSetDevice(device)) != hipSuccess) return host_hip_fail(e, "hipSetDevice");
    b40c_scan_enactor *en = new b40c_scan_enactor();
    en->device = device;
    if ((e = hipStreamCreateWithFlags(&en->stream, hipStreamNonBlocking)) != hipSuccess ||
        (e = hipEventCreate(&en->ev0)) != hipSuccess || (e = hipEventCreate(&en->ev1)) != hipSuccess ||
        (e = en->chain.init(device)) != hipSuccess ||
        (e = take_pinned_word(&en->h_word)) != hipSuccess ||
        (e = hipHostGetDevicePointer(reinterpret_cast<void **>(&en->h_word_dev), en->h_word, 0)) != hipSuccess) {
        b40c_scan_enactor_destroy(en);
        return host_hip_fail(e, "create scan enactor");
    }
    *out = en;
    return BFS_OK;
}

void b40c_scan_enactor_destroy(b40c_scan_enactor *e)
{
    if (!e) return;
    (void) hipSetDevice(e->device);
    if (e->stream) (void) hipStreamSynchronize(e->stream);
    e->chain.release();
    if (e->h_word) give_pinned_word(e->h_word);
    if (e->ev0) (void) hipEventDestroy(e->ev0);
    if (e->ev1) (void) hipEventDestroy(e->ev1);
    if (e->stream) (void) hipStreamDestroy(e->stream);
    delete e;
}

bfs_status b40c_scan(b40c_scan_enactor *e, const uint32_t *d_in, uint32_t *d_out, int64_t n, int32_t exclusive,
                     uint32_t *h_total)
{
    if (!e || n < 0 || (n > 0 && (!d_in || !d_out))) return host_fail(BFS_ERR_INVALID_ARG, "invalid scan arguments");
    if (n > ((int64_t) 1 << 40)) return host_fail(BFS_ERR_INVALID_ARG, "scan longer than 2^40 items");
    hipError_t r;
    if ((r = hipSetDevice(e->device)) != hipSuccess) return host_hip_fail(r, "hipSetDevice");
    if (n == 0) {
        if (h_total) *h_total = 0;
        e->last_ms = 0.f;
        return BFS_OK;
    }
    ChainArgs c;
    if ((r = e->chain.prepare(n, scan_tile_items(n), &c, e->stream)) != hipSuccess)
        return host_hip_fail(r, "scan status storage");
    if ((r = hipEventRecord(e->ev0, e->stream)) != hipSuccess) return host_hip_fail(r, "record");
    if ((r = launch_scan_u32(d_in, d_out, n, exclusive != 0, c, h_total ? e->h_word_dev : nullptr, e->stream)) !=
        hipSuccess)
        return host_hip_fail(r, "launch scan");
    bfs_status st = timed_sync(e);
    if (st != BFS_OK) return st;
    if (h_total) *h_total = *static_cast<volatile uint32_t *>(e->h_word);
    return BFS_OK;
}

bfs_status b40c_copy_if(b40c_scan_enactor *e, const uint32_t *d_in, uint32_t *d_out, int64_t n, b40c_select_op op,
                        uint32_t comparand, int64_t *h_num_compacted, uint32_t *d_num_compacted)
{
    if (!e || n < 0 || (n > 0 && (!d_in || !d_out)) || op < B40C_SELECT_LESS || op > B40C_SELECT_NONNEGATIVE)
        return host_fail(BFS_ERR_INVALID_ARG, "invalid copy-if arguments");
    if (n > (int64_t) UINT32_MAX) return host_fail(BFS_ERR_INVALID_ARG, "copy-if longer than 2^32 - 1 items");
    hipError_t r;
    if ((r = hipSetDevice(e->device)) != hipSuccess) return host_hip_fail(r, "hipSetDevice");
    if (n == 0) {
        if (h_num_compacted) *h_num_compacted = 0;
        if (d_num_compacted && (r = hipMemsetAsync(d_num_compacted, 0, sizeof(uint32_t), e->stream)) != hipSuccess)
            return host_hip_fail(r, "clear count");
        if ((r = hipStreamSynchronize(e->stream)) != hipSuccess) return host_hip_fail(r, "synchronize");
        e->last_ms = 0.f;
        return BFS_OK;
    }
    ChainArgs c;
    if ((r = e->chain.prepare(n, copy_if_tile_items(n), &c, e->stream)) != hipSuccess)
        return host_hip_fail(r, "copy-if status storage");
    if ((r = hipEventRecord(e->ev0, e->stream)) != hipSuccess) return host_hip_fail(r, "record");
    if ((r = launch_copy_if_u32(d_in, d_out, n, (int) op, comparand, c, d_num_compacted,
                                h_num_compacted ? e->h_word_dev : nullptr, e->stream)) != hipSuccess)
        return host_hip_fail(r, "launch copy-if");
    bfs_status st = timed_sync(e);
    if (st != BFS_OK) return st;
    if (h_num_compacted) *h_num_compacted = *static_cast<volatile uint32_t *>(e->h_word);
    return BFS_OK;
}

bfs_status b40c_scan_noalloc(int32_t device, const uint32_t *d_in, uint32_t *d_out, int64_t n, int32_t exclusive,
                             uint32_t *d_total, void *stream)
{
    if (n < 0 || (n > 0 && (!d_in || !d_out))) return host_fail(BFS_ERR_INVALID_ARG, "invalid scan arguments");
    if (n > kNoAllocMaxItems)
        return host_fail(BFS_ERR_INVALID_ARG, "scan longer than the allocation-free limit of 2^26 items");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return host_fail(BFS_ERR_NO_DEVICE, "no HIP device");
    if (device < 0 || device >= count || device >= kNoAllocDevices)
        return host_fail(BFS_ERR_INVALID_ARG, "device ordinal out of range");
    hipError_t r;
    if ((r = hipSetDevice(device)) != hipSuccess) return host_hip_fail(r, "hipSetDevice");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (n == 0) {
        if (d_total) {
            hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, d_total, 1, 0u);
            if ((r = hipGetLastError()) != hipSuccess) return host_hip_fail(r, "clear scan total");
        }
        return BFS_OK;
    }
    unsigned long long *words = nullptr;
    if ((r = noalloc_scratch(device, &words)) != hipSuccess) return host_hip_fail(r, "scan scratch address");
    ChainArgs c;
    const int tile_items = scan_tile_items(n);
    c.tiles = (n + tile_items - 1) / tile_items;
    c.status = words + kNoAllocStatus;
    c.tile_counter = words;
    c.epoch = 0;
    const unsigned clear_blocks = (unsigned) std::min<long long>((c.tiles + kThreads - 1) / kThreads, 64);
    hipLaunchKernelGGL(noalloc_clear_kernel, dim3(clear_blocks), dim3(kThreads), 0, st, words, c.tiles);
    if ((r = hipGetLastError()) != hipSuccess) return host_hip_fail(r, "launch scratch clear");
    if ((r = launch_scan_u32(d_in, d_out, n, exclusive != 0, c, d_total, st)) != hipSuccess)
        return host_hip_fail(r, "launch scan");
    return BFS_OK;
}

bfs_status b40c_scan_last_ms(const b40c_scan_enactor *e, double *ms)
{
    if (!e || !ms) return host_fail(BFS_ERR_INVALID_ARG, "null argument");
    *ms = e->last_ms;
    return BFS_OK;
}

}  // extern "C"
