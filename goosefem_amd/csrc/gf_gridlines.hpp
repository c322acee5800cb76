// Which line of a grid (a column or a row, one direction at a time) each thread of a tile of gf_gridmg.hip
// stands for.  Host and device: the kernels index their vectors with it, and its range is checked on the host.
#pragma once

#include <hip/hip_runtime.h>

namespace gf {

// the wrapped index of a line at most one period out of range, or -1 outside an unwrapped direction
__host__ __device__ inline int wrap_line(int f, int m, int per)
{
    if (f < 0) return per ? f + m : -1;
    if (f >= m) return per ? f - m : -1;
    return f;
}

// Line of lane `lane` of tile `block` of W lanes, of which the inner W - 2 H own a line each.
template <int W, int H>
__host__ __device__ inline int tile_raw(int block, int lane)
{
    return block * (W - 2 * H) + lane - H;
}

// ... in [0, m), or -1 outside an unwrapped direction.  Every lane's line is the true one, also where the
// tile is wider than a wrapped grid.
template <int W, int H>
__host__ __device__ inline int tile_line(int block, int lane, int m, int per)
{
    int f = tile_raw<W, H>(block, lane);
    if (per && m < 2 * W) {
        f %= m;
        return f < 0 ? f + m : f;
    }
    return wrap_line(f, m, per);
}

// ... where only the owned lines and the ring of one around them are used: the lanes beyond that ring stand
// for any line in range, without tile_line's division (a third of the small kernels' time).
template <int W, int H>
__host__ __device__ inline int tile_line_ring(int block, int lane, int m, int per)
{
    const int f = wrap_line(tile_raw<W, H>(block, lane), m, per);
    return f < m ? f : m - 1;
}

} // namespace gf
