// b40c_scan_internal.hpp -- host launchers of the single-pass scan,
// compaction and sort kernels, shared by the scan C ABI (b40c_scan.hip) and
// the device CSR builder (b40c_csr_build.hip).  Not installed.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "b40c_primitives.hpp"

namespace b40c_hip {

constexpr int kScanThreads = 512;

// Items per tile of a scan (copy-if) of n items.
int scan_tile_items(long long n);
int copy_if_tile_items(long long n);

// Arguments of one chained (decoupled look-back) launch.
struct ChainArgs {
    unsigned long long *status;        // one word per tile
    unsigned long long *tile_counter;  // launch-order tile indices; zero before and after every launch
    unsigned epoch;                    // tags this launch's status words
    long long tiles;                   // tiles (= workgroups) of the launch
};

// Device storage of the chained launches of one owner (an enactor or a
// builder), used by one host thread and one stream at a time.
struct ChainState {
    int device = 0;
    unsigned long long *d_counter = nullptr;  // followed by 4 scratch words (d_word)
    uint32_t *d_word = nullptr;
    unsigned long long *d_status = nullptr;
    long long capacity = 0;                   // status words allocated
    unsigned epoch = 0;

    hipError_t init(int dev);
    // Status words and a fresh epoch for a launch over `items` in tiles of
    // tile_items; every launch of a state is on the same stream.  (The tile
    // counter is cleared before the first one alone: the workgroup that takes
    // a launch's last tile sets it back to zero, prim::take_tile.)
    hipError_t prepare(long long items, int tile_items, ChainArgs *c, hipStream_t st);
    void release();
};

hipError_t launch_scan_u32(const uint32_t *in, uint32_t *out, long long n, bool exclusive, const ChainArgs &c,
                           uint32_t *d_total, hipStream_t st);
hipError_t launch_copy_if_u32(const uint32_t *in, uint32_t *out, long long n, int op, uint32_t comparand,
                              const ChainArgs &c, uint32_t *d_count, uint32_t *h_count, hipStream_t st);

namespace prim {

// Tile index from the launch-order counter (every thread calls it).  The
// launch's last tile index goes to the last workgroup to ask, which sets the
// counter back to zero for the next launch.
__device__ __forceinline__ long long take_tile(const ChainArgs &c, long long *s_tile)
{
    if (threadIdx.x == 0) {
        const unsigned long long t = atomicAdd(c.tile_counter, 1ull);
        if (t == (unsigned long long) (c.tiles - 1))
            __hip_atomic_store(c.tile_counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *s_tile = (long long) t;
    }
    __syncthreads();
    return *s_tile;
}

// The tile's exclusive prefix given its aggregate (every thread calls it;
// the result is returned to all).
__device__ __forceinline__ unsigned chain_prefix(const ChainArgs &c, long long tile, unsigned aggregate,
                                                 unsigned *s_prefix)
{
    if (threadIdx.x < kWave) {
        unsigned prefix = 0;
        if (tile == 0) {
            if (threadIdx.x == 0) publish(c.status, tile, c.epoch, kStatePrefix, aggregate);
        } else {
            if (threadIdx.x == 0) publish(c.status, tile, c.epoch, kStateAggregate, aggregate);
            prefix = lookback_prefix(c.status, tile, c.epoch);
            if (threadIdx.x == 0) publish(c.status, tile, c.epoch, kStatePrefix, prefix + aggregate);
        }
        if (threadIdx.x == 0) *s_prefix = prefix;
    }
    __syncthreads();
    return *s_prefix;
}

}  // namespace prim
}  // namespace b40c_hip
