// Work items of the streaming passes (update, scale, widen): one tile of a chunk each; the
// order in which workgroups take them and the grids that launch them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "mi_adamw.h"

namespace {

// The item that workgroup index w takes: in every full group of 8 runs of kRun items, XCD
// w % 8 gets one contiguous run, another one from group to group (a fixed one leaves some
// placements of the update's buffers 3% slower).
template <int kRun>
__host__ __device__ __forceinline__ int64_t item_order(int64_t w, int64_t n_items) {
    static_assert((kRun & (kRun - 1)) == 0, "masks and shifts below");
    constexpr int64_t kGroup = 8 * kRun;
    const int64_t base = w & ~(kGroup - 1);
    if (base + kGroup > n_items) return w;
    const int64_t r = w - base;
    return base + ((r ^ (w >> __builtin_ctzll(kGroup))) & 7) * kRun + (r >> 3);
}

// The items of a launch: chunks of chunk_elems elements, `tiles` tiles each.
struct Items {
    int64_t n;
    int64_t chunk_elems;
    int32_t tiles;
    int32_t shift;    // log2(tiles), or -1
    // Item `it`: its chunk's tensor and row, and the tile's elements.  False past the end of
    // the tensor's last, shorter chunk.
    template <int kTile, class Src>
    __host__ __device__ __forceinline__ bool get(const Src& src, int64_t it, mi_adamw_tensor& t,
                                                 int64_t& begin, int64_t& end,
                                                 int32_t& row) const {
        const int64_t c = shift >= 0 ? it >> shift : it / tiles;
        src.get(c, chunk_elems, t, begin, end, row);
        begin += (it - c * tiles) * kTile;
        if (begin >= end) return false;
        if (end > begin + kTile) end = begin + kTile;
        return true;
    }
};

// The tiles of n_chunks chunks (chunk sizes are multiples of MI_ADAMW_CHUNK_QUANTUM, of which
// every tile size is a divisor).
inline Items items_of(int64_t n_chunks, int64_t chunk_elems, int tile) {
    const int32_t tiles = static_cast<int32_t>(chunk_elems / tile);
    const int32_t shift = (tiles & (tiles - 1)) == 0 ? __builtin_ctz(tiles) : -1;
    return Items{n_chunks * tiles, chunk_elems, tiles, shift};
}

// Workgroups of `threads` lanes for n items, at most max_blocks (0: no bound).
inline unsigned grid_for(int64_t n, int64_t max_blocks, int threads) {
    int64_t g = n;
    if (max_blocks > 0 && g > max_blocks) g = max_blocks;
    if (g > 0x7fffffff / threads) g = 0x7fffffff / threads;
    return static_cast<unsigned>(g);
}

// The update's bound counts lanes in units of 1024, whatever an instance's workgroups are.
constexpr int kBoundThreads = 1024;

inline unsigned update_grid(int64_t n_items, int32_t max_blocks, int threads) {
    return grid_for(n_items, int64_t(max_blocks) * (kBoundThreads / threads), threads);
}

}  // namespace
