// index_map.h -- which tile a workgroup takes. Host code too: the CPU tests compile this file by itself.
#pragma once

namespace eddy {

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on XCD b % 8) and
// each XCD has its own L2. Give workgroups b, b+8, b+16, ... (one XCD) consecutive logical
// tiles, so neighbouring tiles -- which share cache lines at their edges and, for stencils,
// neighbouring planes -- meet in the same L2. Bijective on [0, n).
__host__ __device__ inline int xcd_tile(int b, int n) {
    const int q = n >> 3, r = n & 7;
    const int x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// The same eighths, each walked from its last tile: an XCD starts on what its own L2 (and the
// memory-side cache) still holds of the pass before, and the next pass in forward order on what this
// one leaves. Bijective on [0, n).
__host__ __device__ inline int xcd_tile_back(int b, int n) {
    const int q = n >> 3, r = n & 7;
    const int x = b & 7;
    return (x + 1) * q + (x < r ? x + 1 : r) - 1 - (b >> 3);
}

}  // namespace eddy
