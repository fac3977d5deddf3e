// index_map.h -- which tile a workgroup takes, which cells a lane. Host code too: the CPU tests compile this
// file by itself.
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

// ceil(2^32 / nx): the quotient of an element number below 2^32 by nx as a high product, exact or one
// too large (plane_pair)
__host__ __device__ inline unsigned row_reciprocal(int nx) { return (unsigned)(((1ull << 32) + nx - 1) / nx); }

// The pair of elements r, r + 1 of a field's plane of rows of nx elements (M cells and two ghosts): whether it
// holds an interior cell of rows 1..L, and the x1 and y index of its first element. The second is (i + 1, j), or
// (0, j + 1) past a row's end, which is no interior cell. r may lie past the plane, also by having wrapped below
// its start (the spans of rows shorter than 16 begin there): j is then past L. Unsigned throughout, so that the
// wrapped ones have defined values too.
struct Pair {
    int i, j;
    bool on;
};
__host__ __device__ inline Pair plane_pair(int nx, int M, int L, unsigned r, unsigned rnx) {
    unsigned j = (unsigned)(((unsigned long long)r * rnx) >> 32);
    unsigned i = r - j * (unsigned)nx;
    if (i >= (unsigned)nx) {  // one too large: i wrapped
        --j;
        i += (unsigned)nx;
    }
    return Pair{(int)i, (int)j, j >= 1 && j <= (unsigned)L && i <= (unsigned)M};
}

}  // namespace eddy
