// A gated exclusive scan of int32 values for the list builds, or of two arrays in the same
// launches: tile sums, then tiles applied, each block first adding up the tile sums before its own
// (integer sums: the same whatever the order). Past kScanOwnTiles tiles, where that would read
// more than it saves, one block scans the tile sums in a launch between. Each launch returns at
// once when the build is not running, so a captured update pays two empty launches on steps
// without a rebuild. The first array's tile sums live after the list header in the caller's
// scan_temp buffer, the second's in a scratch array of its own.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace ndn {

constexpr int kScanPerThread = 4;
constexpr int kScanTile = kBlock * kScanPerThread;  // 1024 values per block

// Bytes of the list header at the start of scan_temp; the tile sums follow it. Bytes 64-575 hold
// 64 slots of per-block maxima of the squared displacement at the last reuse check (the bits of
// a nonnegative T, widened to 64 bits), so no slot takes many atomics.
constexpr std::int64_t kHeaderBytes = 1024;
constexpr int kMovedSlots = 64;

struct ListHeader
{
    index_t old_total;  // pair_total before this build: columns past it hold padding
};

__device__ __forceinline__ unsigned long long* moved_slot(ListHeader* header, unsigned block)
{
    return reinterpret_cast<unsigned long long*>(reinterpret_cast<std::uint8_t*>(header) + 64) +
           (block % kMovedSlots);
}

inline std::int64_t scan_tiles(std::int64_t items)
{
    return (items + kScanTile - 1) / kScanTile;
}

inline std::int64_t scan_bytes(std::int64_t items)
{
    return kHeaderBytes + 4 * (scan_tiles(items) + 1);
}

// Tiles up to which a block adds up the tile sums before its own: 16 reads a thread at most.
constexpr std::int64_t kScanOwnTiles = 4096;

// One array of a scan: `count` values, its tile sums (tiles of kScanTile).
struct ScanArray
{
    const index_t* input;
    index_t* output;  // may alias input: each block reads its whole tile before writing it
    std::int64_t count;
    index_t* tile_sums;
};

static __device__ __forceinline__ void scan_tile_sums_body(const ScanArray& a, index_t block)
{
    __shared__ index_t shared[16];
    const std::int64_t base = static_cast<std::int64_t>(block) * kScanTile;
    index_t local = 0;
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k)
    {
        const std::int64_t i = base + threadIdx.x + static_cast<std::int64_t>(k) * kBlock;
        if (i < a.count) local += a.input[i];
    }
    const index_t sum = block_sum(local, shared);
    if (threadIdx.x == 0) a.tile_sums[block] = sum;
}

// The first `first_tiles` blocks take the first array, the rest the second.
static __global__ void __launch_bounds__(kBlock) scan_tile_sums_kernel(
    ScanArray first, ScanArray second, index_t first_tiles, const index_t* rebuild,
    const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const index_t block = static_cast<index_t>(blockIdx.x);
    if (block < first_tiles)
        scan_tile_sums_body(first, block);
    else
        scan_tile_sums_body(second, block - first_tiles);
}

static __global__ void __launch_bounds__(kBlock) scan_tile_prefix_kernel(
    index_t* __restrict__ tile_sums, std::int64_t tiles, const index_t* rebuild,
    const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    __shared__ index_t shared[16];
    index_t carry = 0;
    for (std::int64_t base = 0; base < tiles; base += kScanTile)
    {
        index_t v[kScanPerThread];
        index_t local = 0;
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k)
        {
            const std::int64_t i = base + threadIdx.x * kScanPerThread + k;
            v[k] = i < tiles ? tile_sums[i] : 0;
            local += v[k];
        }
        index_t total;
        index_t running = carry + block_exclusive_sum(local, shared, &total);
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k)
        {
            const std::int64_t i = base + threadIdx.x * kScanPerThread + k;
            if (i < tiles) tile_sums[i] = running;
            running += v[k];
        }
        carry += total;
        __syncthreads();
    }
}

// kOwn: the tile sums are as they were summed and the block adds up those before its own; else
// they are already prefixes.
template <bool kOwn>
__device__ __forceinline__ void scan_apply_body(const ScanArray& a, index_t block)
{
    __shared__ index_t shared[16];
    index_t before = 0;
    if (kOwn)
    {
        index_t local = 0;
        for (index_t k = threadIdx.x; k < block; k += kBlock) local += a.tile_sums[k];
        before = block_sum(local, shared);
    }
    else
        before = a.tile_sums[block];
    const std::int64_t base =
        static_cast<std::int64_t>(block) * kScanTile + threadIdx.x * kScanPerThread;
    index_t v[kScanPerThread];
    index_t local = 0;
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k)
    {
        v[k] = base + k < a.count ? a.input[base + k] : 0;
        local += v[k];
    }
    index_t total;
    index_t running = before + block_exclusive_sum(local, shared, &total);
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k)
    {
        if (base + k < a.count) a.output[base + k] = running;
        running += v[k];
    }
}

template <bool kOwn>
__global__ void __launch_bounds__(kBlock) scan_apply_kernel(ScanArray first, ScanArray second,
                                                            index_t first_tiles,
                                                            const index_t* rebuild,
                                                            const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const index_t block = static_cast<index_t>(blockIdx.x);
    if (block < first_tiles)
        scan_apply_body<kOwn>(first, block);
    else
        scan_apply_body<kOwn>(second, block - first_tiles);
}

// Exclusive scans of one array or of two (second.count 0: none); returns NDN_OK or NDN_ERR_HIP.
inline int exclusive_scans(const ScanArray& first, const ScanArray& second,
                           const index_t* rebuild, const index_t* status, hipStream_t stream)
{
    const std::int64_t tiles = scan_tiles(first.count);
    const std::int64_t more = scan_tiles(second.count);
    const unsigned blocks = static_cast<unsigned>(tiles + more);
    const index_t split = static_cast<index_t>(tiles);
    scan_tile_sums_kernel<<<blocks, kBlock, 0, stream>>>(first, second, split, rebuild, status);
    NDN_LAUNCHED("scan_tile_sums");
    if (std::max(tiles, more) <= kScanOwnTiles)
    {
        scan_apply_kernel<true><<<blocks, kBlock, 0, stream>>>(first, second, split, rebuild,
                                                               status);
        NDN_LAUNCHED("scan_apply");
        return NDN_OK;
    }
    scan_tile_prefix_kernel<<<1, kBlock, 0, stream>>>(first.tile_sums, tiles, rebuild, status);
    NDN_LAUNCHED("scan_tile_prefix");
    if (more > 0)
    {
        scan_tile_prefix_kernel<<<1, kBlock, 0, stream>>>(second.tile_sums, more, rebuild, status);
        NDN_LAUNCHED("scan_tile_prefix");
    }
    scan_apply_kernel<false><<<blocks, kBlock, 0, stream>>>(first, second, split, rebuild, status);
    NDN_LAUNCHED("scan_apply");
    return NDN_OK;
}

// Exclusive scan of `count` values; returns NDN_OK or NDN_ERR_HIP.
inline int exclusive_scan(const index_t* input, index_t* output, std::int64_t count,
                          std::uint8_t* scan_temp, const index_t* rebuild, const index_t* status,
                          hipStream_t stream)
{
    const ScanArray array{input, output, count,
                          reinterpret_cast<index_t*>(scan_temp + kHeaderBytes)};
    return exclusive_scans(array, ScanArray{}, rebuild, status, stream);
}

}  // namespace ndn
