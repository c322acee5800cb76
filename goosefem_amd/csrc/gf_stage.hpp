// LDS staging of contiguous slices, shared by the per-point kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace gf {

// The quadrature kernels read and write per-point / per-element records (dN/dx rows, element
// vectors, tensors) of 8 to 72 bytes.  A workgroup moves its contiguous slice of each array between
// HBM and LDS with full-wave contiguous 16-byte accesses (when the array is 16-byte aligned; element
// by element otherwise) and the threads compute on LDS, so no global access is strided per lane.
template <class T, int NT, int KB>
__device__ inline void stage_in(T* __restrict__ lds, const T* __restrict__ g, int count)
{
    // KB: 16-byte loads in flight per thread before their LDS writes (the call site's typical count)
    constexpr int VW = 16 / static_cast<int>(sizeof(T));
    typedef T V __attribute__((ext_vector_type(VW)));
    int done = 0;
    if ((reinterpret_cast<uintptr_t>(g) & 15) == 0) {
        const int nv = count / VW;
        for (int base = 0; base < nv; base += KB * NT) {
            V r[KB];
            // unconditional loads (an index past the end re-reads the last chunk), so that all KB
            // are issued before the first wait
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                const int i = base + k * NT + threadIdx.x;
                r[k] = reinterpret_cast<const V*>(g)[i < nv ? i : nv - 1];
            }
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                const int i = base + k * NT + threadIdx.x;
                if (i < nv) reinterpret_cast<V*>(lds)[i] = r[k];
            }
        }
        done = nv * VW;
    }
    for (int i = done + threadIdx.x; i < count; i += NT) lds[i] = g[i];
}

template <class T, int NT>
__device__ inline void stage_out(T* __restrict__ g, const T* __restrict__ lds, int count)
{
    constexpr int VW = 16 / static_cast<int>(sizeof(T));
    typedef T V __attribute__((ext_vector_type(VW)));
    int done = 0;
    if ((reinterpret_cast<uintptr_t>(g) & 15) == 0) {
        const int nv = count / VW;
        for (int i = threadIdx.x; i < nv; i += NT)
            __builtin_nontemporal_store(reinterpret_cast<const V*>(lds)[i], reinterpret_cast<V*>(g) + i);
        done = nv * VW;
    }
    for (int i = done + threadIdx.x; i < count; i += NT) g[i] = lds[i];
}

// Rows of W values to rows of pitch W + 1 (an odd number of 8-byte words, so that lanes reading one column
// of consecutive rows fall on different banks); W a multiple of 16 bytes, the slice rows * W values.
template <class T, int NT, int W>
__device__ inline void stage_in_rows(T* __restrict__ lds, const T* __restrict__ g, int rows)
{
    constexpr int VW = 16 / static_cast<int>(sizeof(T));
    static_assert(W % VW == 0, "whole vectors per row");
    typedef T V __attribute__((ext_vector_type(VW)));
    if ((reinterpret_cast<uintptr_t>(g) & 15) == 0) {
        for (int i = threadIdx.x; i < rows * (W / VW); i += NT) {
            const V v = reinterpret_cast<const V*>(g)[i];
            T* d = lds + i * VW + i / (W / VW);
#pragma unroll
            for (int k = 0; k < VW; ++k) d[k] = v[k];
        }
        return;
    }
    for (int i = threadIdx.x; i < rows * W; i += NT) lds[i + i / W] = g[i];
}

} // namespace gf
