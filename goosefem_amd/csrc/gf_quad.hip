// Element quadrature on the device: Element::Quad4::Quadrature (ElementQuad4.h),
// Element::Quad4::QuadraturePlanar (ElementQuad4Planar.h), Element::Hex8::Quadrature
// (ElementHex8.h), with the generic loops of Element.h:892-1229.
//
// FP64 kernels evaluate every expression in the reference's order with no FMA contraction (the
// library is built with -ffp-contract=off), so they reproduce the reference's FP64 bits.  FP32
// kernels run the per-quadrature-point work in single precision on FP32 copies of the geometry.
//
// Launch shape: one thread per (element, quadrature point) or per (element, node); consecutive
// threads touch consecutive elements, so the [nelem, ...] row-major streams are read and written
// in long contiguous runs.
#include <cmath>

#include <type_traits>

#include "gf_internal.hpp"
#include "gf_stage.hpp"

using namespace gf;

struct gf_quad_s {
    int et = 0, nne = 0, ndim = 0, tdim = 0, nip = 0;
    int64_t nelem = 0;
    double thick = 1.0;
    std::vector<double> xi, w, N, dNxi;
    DBuf<double> x, N_d, dNxi_d, w_d, dNx, vol;
    DBuf<float> dNx32, vol32;
    bool have32 = false;
    uint64_t version = 0; // counts update_x: what was derived from dNx or vol is of one version
};

namespace {

constexpr int BS = 256;

inline void shape_functions(int et, int nip, const double* xi, double* N, double* dNxi)
{
    // ElementQuad4.h:287-305, ElementQuad4Planar.h:89-109, ElementHex8.h:265-304
    if (et != GF_HEX8) {
        for (int q = 0; q < nip; ++q) {
            const double x0 = xi[q * 2 + 0], x1 = xi[q * 2 + 1];
            N[q * 4 + 0] = 0.25 * (1.0 - x0) * (1.0 - x1);
            N[q * 4 + 1] = 0.25 * (1.0 + x0) * (1.0 - x1);
            N[q * 4 + 2] = 0.25 * (1.0 + x0) * (1.0 + x1);
            N[q * 4 + 3] = 0.25 * (1.0 - x0) * (1.0 + x1);
            double* d = dNxi + q * 8;
            d[0] = -0.25 * (1.0 - x1);
            d[2] = +0.25 * (1.0 - x1);
            d[4] = +0.25 * (1.0 + x1);
            d[6] = -0.25 * (1.0 + x1);
            d[1] = -0.25 * (1.0 - x0);
            d[3] = -0.25 * (1.0 + x0);
            d[5] = +0.25 * (1.0 + x0);
            d[7] = +0.25 * (1.0 - x0);
        }
        return;
    }
    static const int s[8][3] = {{-1, -1, -1}, {+1, -1, -1}, {+1, +1, -1}, {-1, +1, -1},
                                {-1, -1, +1}, {+1, -1, +1}, {+1, +1, +1}, {-1, +1, +1}};
    for (int q = 0; q < nip; ++q) {
        const double* x = xi + q * 3;
        for (int m = 0; m < 8; ++m) {
            // 0.125 * (1 +- x0) * (1 +- x1) * (1 +- x2), factors in the reference's order
            double f0 = s[m][0] < 0 ? (1.0 - x[0]) : (1.0 + x[0]);
            double f1 = s[m][1] < 0 ? (1.0 - x[1]) : (1.0 + x[1]);
            double f2 = s[m][2] < 0 ? (1.0 - x[2]) : (1.0 + x[2]);
            N[q * 8 + m] = 0.125 * f0 * f1 * f2;
            dNxi[q * 24 + m * 3 + 0] = (s[m][0] < 0 ? -0.125 : +0.125) * f1 * f2;
            dNxi[q * 24 + m * 3 + 1] = (s[m][1] < 0 ? -0.125 : +0.125) * f0 * f2;
            dNxi[q * 24 + m * 3 + 2] = (s[m][2] < 0 ? -0.125 : +0.125) * f0 * f1;
        }
    }
}

inline void default_rule(int et, int rule, std::vector<double>& xi, std::vector<double>& w)
{
    const double a = rule == GF_NODAL ? 1.0 : 1.0 / std::sqrt(3.0);
    if (et != GF_HEX8) {
        const int s[4][2] = {{-1, -1}, {+1, -1}, {+1, +1}, {-1, +1}};
        xi.resize(8);
        w.assign(4, 1.0);
        for (int q = 0; q < 4; ++q)
            for (int d = 0; d < 2; ++d) xi[q * 2 + d] = s[q][d] < 0 ? -a : +a;
    }
    else {
        const int s[8][3] = {{-1, -1, -1}, {+1, -1, -1}, {+1, +1, -1}, {-1, +1, -1},
                             {-1, -1, +1}, {+1, -1, +1}, {+1, +1, +1}, {-1, +1, +1}};
        xi.resize(24);
        w.assign(8, 1.0);
        for (int q = 0; q < 8; ++q)
            for (int d = 0; d < 3; ++d) xi[q * 3 + d] = s[q][d] < 0 ? -a : +a;
    }
}

// ---- geometry: compute_dN ----------------------------------------------------------------------
// ElementQuad4.h:493-532, ElementQuad4Planar.h:280-319 (x thick), Element.h:1178-1229 (Hex8, with
// the chain rule over j)

// dN/dx [4][2] and det J of one Quad4 point.  Shared by the set-up kernel and the kernels that recompute
// the geometry, so all produce the same bits.
__device__ inline void quad4_point_geometry(const double* __restrict__ xe, const double* __restrict__ g, double* o,
                                            double& det)
{
    double J00 = g[0] * xe[0] + g[2] * xe[2] + g[4] * xe[4] + g[6] * xe[6];
    double J01 = g[0] * xe[1] + g[2] * xe[3] + g[4] * xe[5] + g[6] * xe[7];
    double J10 = g[1] * xe[0] + g[3] * xe[2] + g[5] * xe[4] + g[7] * xe[6];
    double J11 = g[1] * xe[1] + g[3] * xe[3] + g[5] * xe[5] + g[7] * xe[7];
    det = J00 * J11 - J01 * J10; // detail.h:17-37
    double I00 = J11 / det, I01 = -1.0 * J01 / det, I10 = -1.0 * J10 / det, I11 = J00 / det;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        o[m * 2 + 0] = I00 * g[m * 2 + 0] + I01 * g[m * 2 + 1];
        o[m * 2 + 1] = I10 * g[m * 2 + 0] + I11 * g[m * 2 + 1];
    }
}

__global__ void k_compute_dN_quad4(int64_t n, int nip, int planar, double thick, const double* __restrict__ x,
                                   const double* __restrict__ dNxi, const double* __restrict__ w,
                                   double* __restrict__ dNx, double* __restrict__ vol)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / nip;
    int q = static_cast<int>(t - e * nip);
    double det;
    quad4_point_geometry(x + e * 8, dNxi + q * 8, dNx + t * 8, det);
    vol[t] = planar ? w[q] * det * thick : w[q] * det;
}

// dN/dx [8][3] and det J of one Hex8 point: J = dN/dxi^T x_e, its cofactor inverse (detail.h:40-70),
// dN/dx = J^-1 dN/dxi, in the generic compute_dN order (Element.h:1178-1229, with the Q1 chain rule
// corrected).  Shared by the set-up kernel and the gradient kernel that recomputes the geometry, so
// both produce the same bits.
__device__ inline void hex8_point_geometry(const double* __restrict__ xe, const double* __restrict__ g, double* o,
                                           double& det)
{
    double A[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) A[i][j] = 0.0;
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) A[i][j] += g[m * 3 + i] * xe[m * 3 + j];
    det = (A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0] + A[0][2] * A[1][0] * A[2][1]) -
          (A[0][2] * A[1][1] * A[2][0] + A[0][1] * A[1][0] * A[2][2] + A[0][0] * A[1][2] * A[2][1]);
    double B[3][3];
    B[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) / det;
    B[0][1] = (A[0][2] * A[2][1] - A[0][1] * A[2][2]) / det;
    B[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) / det;
    B[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) / det;
    B[1][1] = (A[0][0] * A[2][2] - A[0][2] * A[2][0]) / det;
    B[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) / det;
    B[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) / det;
    B[2][1] = (A[0][1] * A[2][0] - A[0][0] * A[2][1]) / det;
    B[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) / det;
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            double s = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j) s += B[i][j] * g[m * 3 + j];
            o[m * 3 + i] = s;
        }
}

__global__ void k_compute_dN_hex8(int64_t n, int nip, const double* __restrict__ x, const double* __restrict__ dNxi,
                                  const double* __restrict__ w, double* __restrict__ dNx, double* __restrict__ vol)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / nip;
    int q = static_cast<int>(t - e * nip);
    double det;
    hex8_point_geometry(x + e * 24, dNxi + q * 24, dNx + t * 24, det);
    vol[t] = w[q] * det;
}

// The FP32 copies of a Hex8 quadrature's dN/dx and dV: formed in FP64 again from the coordinates (192 bytes
// per element) and rounded once, which is the stored FP64 value rounded (1,600 bytes per element to read);
// the rows leave through LDS as one contiguous stream.
constexpr int GB32 = 256; // points per workgroup

inline size_t geo32_lds_bytes(int nip)
{
    return static_cast<size_t>(GB32) * 24 * 4 + (GB32 / nip + 2) * 25 * 8 + static_cast<size_t>(nip) * 25 * 8;
}

__global__ void __launch_bounds__(GB32) k_geometry32_hex8(int64_t n, int nip, const double* __restrict__ x,
                                                          const double* __restrict__ dNxi,
                                                          const double* __restrict__ w, float* __restrict__ dNx,
                                                          float* __restrict__ vol)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float* s_o = reinterpret_cast<float*>(smem);                // [GB32][24]
    double* s_x = reinterpret_cast<double*>(s_o + GB32 * 24);   // [GB32 / nip + 2][25]
    double* s_d = s_x + (GB32 / nip + 2) * 25;                  // [nip][25]
    const int64_t t0 = blockIdx.x * static_cast<int64_t>(GB32);
    const int nq = static_cast<int>(min<int64_t>(GB32, n - t0));
    const int64_t e0 = t0 / nip, e1 = (t0 + nq - 1) / nip;
    stage_in_rows<double, GB32, 24>(s_x, x + e0 * 24, static_cast<int>(e1 - e0 + 1));
    for (int i = threadIdx.x; i < nip * 24; i += GB32) s_d[i + i / 24] = dNxi[i];
    __syncthreads();
    if (threadIdx.x < nq) {
        const int p = static_cast<int>(t0 - e0 * nip) + threadIdx.x, el = p / nip, q = p - el * nip;
        double gd[24], det;
        hex8_point_geometry(s_x + el * 25, s_d + q * 25, gd, det);
#pragma unroll
        for (int k = 0; k < 24; ++k) s_o[threadIdx.x * 24 + k] = static_cast<float>(gd[k]);
        vol[t0 + threadIdx.x] = static_cast<float>(w[q] * det);
    }
    __syncthreads();
    stage_out<float, GB32>(dNx + t0 * 24, s_o, nq * 24);
}

__global__ void k_to_f32(int64_t n, const double* __restrict__ a, float* __restrict__ b)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t < n) b[t] = static_cast<float>(a[t]);
}

// ---- gradients: mode 0 GradN_vector, 1 GradN_vector_T, 2 SymGradN_vector -------------------------

// GradN_vector (mode 0), GradN_vector_T (1), SymGradN_vector (2): 2-D node vectors (Quad4 tdim 2 /
// planar tdim 3, ElementQuad4.h:348-434, ElementQuad4Planar.h:129-221) and Hex8 (the generic loops of
// Element.h:924-1022), in the reference's expression order.  A workgroup of QB threads owns QB
// consecutive points (e, q) and moves its slices through LDS.
//
// Quad4: bound by HBM.  dN/dx of a point is formed from the 64 bytes of element coordinates with
// quad4_point_geometry, the function that produced the stored ones (FP32: the FP64 dN/dx rounded once, as
// the stored FP32 copy is), so the results are the stored geometry's bit for bit, for 416 instead of 608
// bytes per element (planar, FP64; FP32 240 instead of 304).  2.0 M planar elements: 217 -> 137 us FP64 (6.1 TB/s), 102 -> 93 us
// FP32.
template <class T, int TD, int mode>
__global__ void __launch_bounds__(256) k_grad_2d_x(int64_t n, int nip, const double* __restrict__ x,
                                                   const double* __restrict__ dNxi, const T* __restrict__ elemvec,
                                                   T* __restrict__ qtensor)
{
    constexpr int QB = 256;
    extern __shared__ __align__(16) unsigned char smem[];
    const int nemax = QB / nip + 2;
    double* s_x = reinterpret_cast<double*>(smem);  // [nemax][8]
    T* s_u = reinterpret_cast<T*>(s_x + nemax * 8); // [nemax][8]
    T* s_o = s_u + nemax * 8;                        // [QB][TD TD]
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * QB;
    const int nq = static_cast<int>(min<int64_t>(QB, n - t0));
    const int64_t e0 = t0 / nip, e1 = (t0 + nq - 1) / nip;
    const int ne = static_cast<int>(e1 - e0 + 1);
    stage_in<double, QB, 1>(s_x, x + e0 * 8, ne * 8);
    stage_in<T, QB, 1>(s_u, elemvec + e0 * 8, ne * 8);
    __syncthreads();
    if (threadIdx.x < nq) {
        // point t0 + threadIdx.x: t0 = e0 nip + (t0 % nip), so the division is a 32-bit one
        const int p = static_cast<int>(t0 - e0 * nip) + threadIdx.x, el = p / nip, q = p - el * nip;
        double gd[8], det;
        quad4_point_geometry(s_x + el * 8, dNxi + q * 8, gd, det);
        T g[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) g[k] = static_cast<T>(gd[k]);
        const T* u = s_u + el * 8;
        T a00 = g[0] * u[0] + g[2] * u[2] + g[4] * u[4] + g[6] * u[6];
        T a01 = g[0] * u[1] + g[2] * u[3] + g[4] * u[5] + g[6] * u[7];
        T a10 = g[1] * u[0] + g[3] * u[2] + g[5] * u[4] + g[7] * u[6];
        T a11 = g[1] * u[1] + g[3] * u[3] + g[5] * u[5] + g[7] * u[7];
        T r[TD * TD];
#pragma unroll
        for (int k = 0; k < TD * TD; ++k) r[k] = T(0);
        if constexpr (mode == 0) {
            r[0] = a00;
            r[1] = a01;
            r[TD] = a10;
            r[TD + 1] = a11;
        }
        else if constexpr (mode == 1) {
            r[0] = a00;
            r[TD] = a01;
            r[1] = a10;
            r[TD + 1] = a11;
        }
        else {
            r[0] = a00;
            r[TD + 1] = a11;
            r[1] = T(0.5) * (g[0] * u[1] + g[2] * u[3] + g[4] * u[5] + g[6] * u[7] + g[1] * u[0] + g[3] * u[2] +
                             g[5] * u[4] + g[7] * u[6]);
            r[TD] = r[1];
        }
        T* o = s_o + threadIdx.x * TD * TD;
#pragma unroll
        for (int k = 0; k < TD * TD; ++k) o[k] = r[k];
    }
    __syncthreads();
    stage_out<T, QB>(qtensor + t0 * TD * TD, s_o, nq * TD * TD);
}

inline size_t grad2x_lds_bytes(int nip, int td, size_t sz)
{
    const size_t ne = 256 / nip + 2;
    return ne * 8 * 8 + ne * 8 * sz + 256 * static_cast<size_t>(td * td) * sz;
}

// Hex8 with the stored geometry: rules of so few points that the coordinates of a workgroup's elements
// outgrow LDS.  LDS holds the points' dN/dx rows [QB][24], element vectors and output tensors.
inline size_t grad3_lds_bytes(int qb, int nip, size_t sz)
{
    return (static_cast<size_t>(qb) * 24 + static_cast<size_t>(qb) * 9 + (qb / nip + 2) * 24) * sz;
}

template <class T, int mode>
__global__ void __launch_bounds__(128) k_grad_3d_lds(int64_t n, int nip, const T* __restrict__ dNx,
                                                     const T* __restrict__ elemvec, T* __restrict__ qtensor)
{
    constexpr int QB = 128;
    extern __shared__ __align__(16) unsigned char smem[];
    T* s_o = reinterpret_cast<T*>(smem); // [QB][9]
    T* s_g = s_o + QB * 9;           // [QB][24]
    T* s_u = s_g + QB * 24;           // [elements][24]
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * QB;
    const int nq = static_cast<int>(min<int64_t>(QB, n - t0));
    const int64_t e0 = t0 / nip, e1 = (t0 + nq - 1) / nip;
    stage_in<T, QB, 24 / (16 / sizeof(T))>(s_g, dNx + t0 * 24, nq * 24);
    stage_in<T, QB, 1>(s_u, elemvec + e0 * 24, static_cast<int>(e1 - e0 + 1) * 24);
    __syncthreads();
    if (threadIdx.x < nq) {
        const int64_t e = (t0 + threadIdx.x) / nip;
        const T* u = s_u + (e - e0) * 24;
        const T* g = s_g + threadIdx.x * 24;
        T r[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) r[k] = T(0);
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if constexpr (mode == 0) r[i * 3 + j] += g[m * 3 + i] * u[m * 3 + j];
                    else if constexpr (mode == 1) r[j * 3 + i] += g[m * 3 + i] * u[m * 3 + j];
                    else {
                        T h = T(0.5) * g[m * 3 + i] * u[m * 3 + j];
                        r[i * 3 + j] += h;
                        r[j * 3 + i] += h;
                    }
                }
        T* o = s_o + threadIdx.x * 9;
#pragma unroll
        for (int k = 0; k < 9; ++k) o[k] = r[k];
    }
    __syncthreads();
    stage_out<T, QB>(qtensor + t0 * 9, s_o, nq * 9);
}

// Hex8 gradients with the geometry recomputed: the stored dN/dx of a Hex8 quadrature is 1536 bytes
// per element against 192 bytes of element coordinates, so this kernel reads the coordinates (kept by
// the quadrature) and forms each point's dN/dx with hex8_point_geometry, the function that produced the
// stored ones: the results are bit-identical to the stored-geometry form (FP32: the FP64 dN/dx rounded
// once, as the stored FP32 copy is).  A workgroup of QB threads owns QB consecutive points; LDS holds
// the coordinates and element vectors of the elements they span, the reference-element gradients and
// the output tensors.
constexpr int QB3 = 256;

inline size_t grad3x_lds_bytes(int nip, size_t sz)
{
    const size_t ne = QB3 / nip + 2;
    return static_cast<size_t>(QB3) * 9 * sz + ne * 24 * sz + ne * 24 * 8 + static_cast<size_t>(nip) * 24 * 8;
}

template <class T, int mode>
__global__ void __launch_bounds__(QB3) k_grad_3d_x(int64_t n, int nip, const double* __restrict__ x,
                                                   const double* __restrict__ dNxi, const T* __restrict__ elemvec,
                                                   T* __restrict__ qtensor)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * QB3;
    const int nq = static_cast<int>(min<int64_t>(QB3, n - t0));
    const int64_t e0 = t0 / nip, e1 = (t0 + nq - 1) / nip;
    const int ne = static_cast<int>(e1 - e0 + 1), nemax = QB3 / nip + 2;
    T* s_o = reinterpret_cast<T*>(smem);       // [QB3][9]
    T* s_u = s_o + QB3 * 9;                      // [nemax][24]
    double* s_x = reinterpret_cast<double*>(s_u + nemax * 24); // [nemax][24]
    double* s_d = s_x + nemax * 24;              // [nip][24]
    stage_in<T, QB3, 1>(s_u, elemvec + e0 * 24, ne * 24);
    stage_in<double, QB3, 1>(s_x, x + e0 * 24, ne * 24);
    for (int i = threadIdx.x; i < nip * 24; i += QB3) s_d[i] = dNxi[i];
    __syncthreads();
    if (threadIdx.x < nq) {
        const int p = static_cast<int>(t0 - e0 * nip) + threadIdx.x, el = p / nip, q = p - el * nip;
        double gd[24], det;
        hex8_point_geometry(s_x + el * 24, s_d + q * 24, gd, det);
        T g[24];
#pragma unroll
        for (int k = 0; k < 24; ++k) g[k] = static_cast<T>(gd[k]);
        const T* u = s_u + el * 24;
        T r[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) r[k] = T(0);
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    if constexpr (mode == 0) r[i * 3 + j] += g[m * 3 + i] * u[m * 3 + j];
                    else if constexpr (mode == 1) r[j * 3 + i] += g[m * 3 + i] * u[m * 3 + j];
                    else {
                        T h = T(0.5) * g[m * 3 + i] * u[m * 3 + j];
                        r[i * 3 + j] += h;
                        r[j * 3 + i] += h;
                    }
                }
        T* o = s_o + threadIdx.x * 9;
#pragma unroll
        for (int k = 0; k < 9; ++k) o[k] = r[k];
    }
    __syncthreads();
    stage_out<T, QB3>(qtensor + t0 * 9, s_o, nq * 9);
}

// ---- interpolation / integration ----------------------------------------------------------------

// InterpQuad_vector: Quad4 override for n = 2 (ElementQuad4.h:324-346) has the same order as the
// generic loop (Element.h:892-922) when starting from 0
__global__ void k_interp(int64_t n, int nip, int nne, int nv, const double* __restrict__ N,
                         const double* __restrict__ elemvec, double* __restrict__ qvector)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / nip;
    int q = static_cast<int>(t - e * nip);
    const double* f = elemvec + e * nne * nv;
    for (int i = 0; i < nv; ++i) {
        double s = 0.0;
        for (int m = 0; m < nne; ++m) s += N[q * nne + m] * f[m * nv + i];
        qvector[t * nv + i] = s;
    }
}

// Int_N_vector_dV (Element.h:1024-1055): thread per (e, m)
__global__ void k_int_N_vector(int64_t n, int nip, int nne, int nv, const double* __restrict__ N,
                               const double* __restrict__ vol, const double* __restrict__ qvector,
                               double* __restrict__ elemvec)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / nne;
    int m = static_cast<int>(t - e * nne);
    for (int i = 0; i < nv; ++i) {
        double s = 0.0;
        for (int q = 0; q < nip; ++q) s += N[q * nne + m] * qvector[(e * nip + q) * nv + i] * vol[e * nip + q];
        elemvec[t * nv + i] = s;
    }
}

// Int_N_scalar_NT_dV (ElementQuad4.h:436-464, ElementQuad4Planar.h:223-251, ElementHex8.h:323-352):
// thread per (e, m, n) writes the nd x nd block (diagonal = accumulated scalar, else 0)
__global__ void k_int_N_scalar(int64_t n, int nip, int nne, int nd, const double* __restrict__ N,
                               const double* __restrict__ vol, const double* __restrict__ qscalar,
                               double* __restrict__ elemmat)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / (nne * nne);
    int mn = static_cast<int>(t - e * nne * nne);
    int m = mn / nne, nn = mn - m * nne;
    double s = 0.0;
    for (int q = 0; q < nip; ++q) s += N[q * nne + m] * qscalar[e * nip + q] * N[q * nne + nn] * vol[e * nip + q];
    int K = nne * nd;
    double* M = elemmat + e * K * K;
    for (int i = 0; i < nd; ++i)
        for (int j = 0; j < nd; ++j) M[(m * nd + i) * K + nn * nd + j] = (i == j) ? s : 0.0;
}

// Int_gradN_dot_tensor2_dV: thread per (e, m)
template <class T, int ND, int TD>
__global__ void k_int_tensor2(int64_t n, int nip, int nne, const T* __restrict__ dNx, const T* __restrict__ vol,
                              const T* __restrict__ qtensor, T* __restrict__ elemvec)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / nne;
    int m = static_cast<int>(t - e * nne);
    T f[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) f[j] = T(0);
    for (int q = 0; q < nip; ++q) {
        const T* g = dNx + ((e * nip + q) * nne + m) * ND;
        const T* s = qtensor + (e * nip + q) * TD * TD;
        T v = vol[e * nip + q];
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            T a = g[0] * s[0 * TD + j] + g[1] * s[1 * TD + j];
            if (ND == 3) a = a + g[2] * s[2 * TD + j];
            f[j] += a * v;
        }
    }
#pragma unroll
    for (int j = 0; j < ND; ++j) elemvec[t * ND + j] = f[j];
}

// The same integral with the geometry recomputed from the element coordinates, by the set-up's own
// functions (bit-identical; FP32: dN/dx and dV rounded once, as the stored FP32 copies are).  A workgroup
// owns PB / nip whole elements; one thread per point forms the point's contributions
// (dN/dx(m, :) . sigma(:, j)) dV of every node from registers, then one thread per (element, node) adds
// its points' contributions in order, from LDS: the order of k_int_tensor2, and the point's data is read
// once instead of once per node.
// Bound: HBM (Quad4; Hex8 FP64 close to FP64 issue).  Bytes per element, stored -> recomputed geometry:
// Quad4 planar FP64 640 -> 416, FP32 320 -> 240; Hex8 FP64 2,368 -> 960, FP32 1,184 -> 576.
// 2.0 M planar Quad4: 239 -> 142 us FP64 (5.9 TB/s), 128 -> 96 us FP32; 395 k Hex8: 178 -> 153 us FP64, 91 ->
// 85 us FP32 (the stored FP32 geometry, below).
constexpr int PB2 = 256; // Quad4 points per workgroup

template <class T, int TD>
__global__ void __launch_bounds__(PB2) k_int_tensor2_q4(int64_t nelem, int nip, int planar, double thick,
                                                        const double* __restrict__ x, const double* __restrict__ dNxi,
                                                        const double* __restrict__ w, const T* __restrict__ qtensor,
                                                        T* __restrict__ elemvec)
{
    constexpr int ROW = TD * TD > 8 ? TD * TD : 8; // a point's contributions overwrite its tensor
    constexpr int TB = TD * TD == ROW ? 0 : PB2 * ROW; // (TD = 2: the tensors lie behind them)
    extern __shared__ __align__(16) unsigned char smem[];
    const int EB = PB2 / nip; // elements of the workgroup
    T* s_c = reinterpret_cast<T*>(smem);                        // [PB2][ROW]
    T* s_s = s_c + TB;                                          // [PB2][TD TD]
    double* s_x = reinterpret_cast<double*>(s_s + PB2 * TD * TD); // [EB][8], then the element vectors
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * EB;
    const int ne = static_cast<int>(min<int64_t>(EB, nelem - e0)), np = ne * nip;
    stage_in<T, PB2, (TD * TD * sizeof(T) + 15) / 16>(s_s, qtensor + e0 * nip * TD * TD, np * TD * TD);
    stage_in<double, PB2, 1>(s_x, x + e0 * 8, ne * 8);
    __syncthreads();
    if (threadIdx.x < np) {
        const int el = threadIdx.x / nip, q = threadIdx.x - el * nip;
        double gd[8], det;
        quad4_point_geometry(s_x + el * 8, dNxi + q * 8, gd, det);
        const T v = static_cast<T>(planar ? w[q] * det * thick : w[q] * det);
        T s[TD * TD], c[8];
#pragma unroll
        for (int k = 0; k < TD * TD; ++k) s[k] = s_s[threadIdx.x * TD * TD + k];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const T g0 = static_cast<T>(gd[2 * m]), g1 = static_cast<T>(gd[2 * m + 1]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const T a = g0 * s[j] + g1 * s[TD + j];
                c[2 * m + j] = a * v;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) s_c[threadIdx.x * ROW + k] = c[k];
    }
    __syncthreads();
    T* s_o = reinterpret_cast<T*>(s_x);
    for (int t = threadIdx.x; t < ne * 4; t += PB2) {
        const T* c = s_c + (t / 4) * nip * ROW + (t % 4) * 2;
        T f0 = T(0), f1 = T(0);
        for (int q = 0; q < nip; ++q) {
            f0 += c[q * ROW];
            f1 += c[q * ROW + 1];
        }
        s_o[2 * t] = f0;
        s_o[2 * t + 1] = f1;
    }
    __syncthreads();
    stage_out<T, PB2>(elemvec + e0 * 8, s_o, ne * 8);
}

inline size_t int2_q4_lds_bytes(int nip, int td, size_t sz)
{
    return static_cast<size_t>(PB2) * (td == 3 ? 9 : 12) * sz + static_cast<size_t>(PB2 / nip) * 8 * 8;
}

constexpr int PB3 = 128; // Hex8 points per workgroup

// FP32 reads the stored FP32 geometry (each thread its point's 96 bytes; gx, gv), FP64 the coordinates
// (gx) and weights (gv).
template <class T>
__global__ void __launch_bounds__(PB3) k_int_tensor2_h8(int64_t nelem, int nip, const T* __restrict__ gx,
                                                        const double* __restrict__ dNxi, const T* __restrict__ gv,
                                                        const T* __restrict__ qtensor, T* __restrict__ elemvec)
{
    constexpr bool STORED = std::is_same_v<T, float>;
    extern __shared__ __align__(16) unsigned char smem[];
    const int EB = PB3 / nip;
    T* s_c = reinterpret_cast<T*>(smem);                  // [PB3][13]: four nodes' contributions at a time
    T* s_s = s_c + PB3 * 13;                              // [PB3][9], then the element vectors [EB][24]
    double* s_x = reinterpret_cast<double*>(s_s + PB3 * 24 / (nip < 2 ? 1 : 2)); // [EB][25] (FP64)
    double* s_d = s_x + EB * 25;                          // [nip][25] (FP64)
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * EB;
    const int ne = static_cast<int>(min<int64_t>(EB, nelem - e0)), np = ne * nip;
    stage_in<T, PB3, (9 * sizeof(T) + 15) / 16>(s_s, qtensor + e0 * nip * 9, np * 9);
    const int el = threadIdx.x / nip, q = threadIdx.x - el * nip;
    T g[24], s[9], v = T(0);
    if constexpr (STORED) {
        typedef float V __attribute__((ext_vector_type(4)));
        const int64_t t = e0 * nip + min(static_cast<int>(threadIdx.x), np - 1);
        const V* row = reinterpret_cast<const V*>(gx + t * 24);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const V r = row[k];
#pragma unroll
            for (int i = 0; i < 4; ++i) g[4 * k + i] = r[i];
        }
        v = gv[t];
    }
    else {
        stage_in_rows<double, PB3, 24>(s_x, gx + e0 * 24, ne);
        for (int i = threadIdx.x; i < nip * 24; i += PB3) s_d[i + i / 24] = dNxi[i];
    }
    __syncthreads();
    if (threadIdx.x < np) {
        if constexpr (!STORED) {
            double det;
            hex8_point_geometry(s_x + el * 25, s_d + q * 25, g, det);
            v = gv[q] * det;
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) s[k] = s_s[threadIdx.x * 9 + k];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads(); // the tensors (h = 0), then the first nodes' contributions (h = 1) are read
        if (threadIdx.x < np) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const T* gm = g + (4 * h + m) * 3;
                    T a = gm[0] * s[j] + gm[1] * s[3 + j];
                    a = a + gm[2] * s[6 + j];
                    s_c[threadIdx.x * 13 + m * 3 + j] = a * v;
                }
        }
        __syncthreads();
        for (int t = threadIdx.x; t < ne * 12; t += PB3) {
            const int e = t / 12, k = t - e * 12;
            const T* c = s_c + e * nip * 13 + k;
            T f = T(0);
            for (int i = 0; i < nip; ++i) f += c[i * 13];
            s_s[e * 24 + 12 * h + k] = f;
        }
    }
    __syncthreads();
    stage_out<T, PB3>(elemvec + e0 * 24, s_s, ne * 24);
}

// FP32 Hex8 from the stored geometry with everything staged: whole-wave streams of dN/dx, dV and the
// tensors, one thread per (element, node) over the points.  The same order of sums.  Taken where the arrays
// leave the caches behind: us with k_int_tensor2_h8 and staged, 110,592 elements 20.9 and 23.5; 394,831: 82.1
// and 82.0; 884,736: 182 and 176; 2,097,152: 441 and 416.
constexpr int EBS = 16; // elements per workgroup
constexpr int64_t H8_STAGED = 400000;

inline size_t int2_h8_staged_lds_bytes(int nip) { return (static_cast<size_t>(EBS) * nip * 34 + EBS * 24) * 4; }

__global__ void __launch_bounds__(EBS * 8) k_int_tensor2_h8_staged(int64_t nelem, int nip, const float* __restrict__ dNx,
                                                                   const float* __restrict__ vol,
                                                                   const float* __restrict__ qtensor,
                                                                   float* __restrict__ elemvec)
{
    constexpr int NT = EBS * 8;
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * EBS;
    const int ne = static_cast<int>(min<int64_t>(EBS, nelem - e0));
    float* s_g = reinterpret_cast<float*>(smem); // [EBS nip][24]
    float* s_s = s_g + EBS * nip * 24;           // [EBS nip][9]
    float* s_o = s_s + EBS * nip * 9;            // [EBS][24]
    float* s_v = s_o + EBS * 24;                 // [EBS nip]
    stage_in<float, NT, 6>(s_g, dNx + e0 * nip * 24, ne * nip * 24);
    stage_in<float, NT, 3>(s_s, qtensor + e0 * nip * 9, ne * nip * 9);
    stage_in<float, NT, 1>(s_v, vol + e0 * nip, ne * nip);
    __syncthreads();
    const int el = threadIdx.x / 8, m = threadIdx.x % 8;
    if (el < ne) {
        float f[3] = {0.0f, 0.0f, 0.0f};
        for (int q = 0; q < nip; ++q) {
            const float *g = s_g + ((el * nip + q) * 8 + m) * 3, *sq = s_s + (el * nip + q) * 9;
            const float v = s_v[el * nip + q];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                float a = g[0] * sq[j] + g[1] * sq[3 + j];
                a = a + g[2] * sq[6 + j];
                f[j] += a * v;
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) s_o[(el * 8 + m) * 3 + j] = f[j];
    }
    __syncthreads();
    stage_out<float, NT>(elemvec + e0 * 24, s_o, ne * 24);
}

// (at least 9 values per point and 24 per element behind the contributions)
inline size_t int2_h8_lds_bytes(int nip, size_t sz)
{
    return static_cast<size_t>(PB3) * 13 * sz + static_cast<size_t>(PB3) * 24 / (nip < 2 ? 1 : 2) * sz +
           (sz == 4 ? 0 : static_cast<size_t>(PB3 / nip) * 25 * 8 + static_cast<size_t>(nip) * 25 * 8);
}

// Int_gradN_dot_tensor4_dot_gradNT_dV FP64 (Element.h:1131-1176): thread per (e, m, n) block
template <int NNE, int ND, int TD>
__global__ void k_int_tensor4_f64(int64_t n, int nip, const double* __restrict__ dNx, const double* __restrict__ vol,
                                  const double* __restrict__ C, double* __restrict__ elemmat)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    int64_t e = t / (NNE * NNE);
    int mn = static_cast<int>(t - e * NNE * NNE);
    int m = mn / NNE, nn = mn - m * NNE;
    double acc[ND][ND];
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int k = 0; k < ND; ++k) acc[j][k] = 0.0;
    for (int q = 0; q < nip; ++q) {
        const double* g = dNx + (e * nip + q) * NNE * ND;
        const double* Cq = C + (e * nip + q) * TD * TD * TD * TD;
        double v = vol[e * nip + q];
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int j = 0; j < ND; ++j)
#pragma unroll
                for (int k = 0; k < ND; ++k)
#pragma unroll
                    for (int l = 0; l < ND; ++l)
                        acc[j][k] += g[m * ND + i] * Cq[((i * TD + j) * TD + k) * TD + l] * g[nn * ND + l] * v;
    }
    constexpr int K = NNE * ND;
    double* Ke = elemmat + e * K * K;
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int k = 0; k < ND; ++k) Ke[(m * ND + j) * K + nn * ND + k] = acc[j][k];
}

// The same integral for Quad4 with four points (planar TD = 3, plain TD = 2), FP64, as one thread per
// (element, node m): per point the products dNx(m, i) C(i, j, k, l) are formed once and used for all
// four column nodes n, in the generic loop's expression and summation order (bit-identical to it).
// A block owns 64 elements.  The whole block first copies the 16 in-plane entries of its 256 points'
// tangents into LDS (a planar point's 81-entry record is read only where it holds them: 8.7 GB of
// HBM reads at 2048^2 against 10.8 GB when each thread loads its own, and 8 % less time); the K_e
// rows then go through the same LDS (rows padded against bank conflicts) and leave as one contiguous
// 16-byte stream: a thread writing its own 128-byte rows directly costs several times the kernel's
// time.  Needs a 16-byte aligned elemmat.
constexpr int T4_EB = 64, T4_KROW = 18;

template <int TD>
__global__ void __launch_bounds__(4 * T4_EB)
    k_int_tensor4_q4_f64(int64_t nelem, const double* __restrict__ dNx, const double* __restrict__ vol,
                         const double* __restrict__ C, double* __restrict__ elemmat)
{
    typedef double dbl2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double sK[4 * T4_EB * T4_KROW]; // staged C [256][16], then K_e rows
    static_assert(T4_KROW >= 16, "the staged tangents must fit");
    const int64_t e0 = blockIdx.x * static_cast<int64_t>(T4_EB);
    const int ne = static_cast<int>(nelem - e0 < T4_EB ? nelem - e0 : T4_EB);
    const int t = threadIdx.x, el = t / 4, m = t % 4;
    {
        // entry r = ((i 2 + j) 2 + k) 2 + l of point p at sK[16 p + r]
        const double* Cb = C + e0 * 4 * TD * TD * TD * TD;
        for (int w = t; w < 64 * ne; w += 4 * T4_EB) {
            const int p = w / 16, r = w % 16, i = r / 8, j = (r / 4) % 2, k = (r / 2) % 2, l = r % 2;
            sK[w] = Cb[p * TD * TD * TD * TD + ((i * TD + j) * TD + k) * TD + l];
        }
    }
    __syncthreads();
    double acc[4][2][2]; // acc[n][j][k] = K(2m + j, 2n + k)
    if (t < 4 * ne) {
        const int64_t e = e0 + el;
#pragma unroll
        for (int nn = 0; nn < 4; ++nn)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int k = 0; k < 2; ++k) acc[nn][j][k] = 0.0;
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            const double* g = dNx + (e * 4 + q) * 8;
            const double* Cq = sK + 16 * (4 * el + q);
            const double v = vol[e * 4 + q];
            double gv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) gv[k] = g[k];
            double gc[2][2][2][2]; // dNx(m, i) * C(i, j, k, l)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int l = 0; l < 2; ++l) gc[i][j][k][l] = gv[m * 2 + i] * Cq[((i * 2 + j) * 2 + k) * 2 + l];
#pragma unroll
            for (int nn = 0; nn < 4; ++nn)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int l = 0; l < 2; ++l) acc[nn][j][k] += gc[i][j][k][l] * gv[nn * 2 + l] * v;
        }
    }
    __syncthreads(); // the staged tangents are consumed
    if (t < 4 * ne) {
        dbl2* row = reinterpret_cast<dbl2*>(sK + T4_KROW * t); // rows 2m, 2m + 1: 16 contiguous doubles
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int nn = 0; nn < 4; ++nn) row[4 * j + nn] = dbl2{acc[nn][j][0], acc[nn][j][1]};
    }
    __syncthreads();
    // the block's K_e are 8 * (4 ne) contiguous 16-byte pieces; piece w is piece w % 8 of row w / 8
    dbl2* K = reinterpret_cast<dbl2*>(elemmat + 64 * e0);
    for (int w = t; w < 32 * ne; w += 4 * T4_EB)
        __builtin_nontemporal_store(reinterpret_cast<const dbl2*>(sK + T4_KROW * (w / 8))[w % 8], K + w);
}

// ---- material ----------------------------------------------------------------------------------

// Linear elastic stress per point.  Bound by HBM (72 + 16 bytes read, 72 written per 3 x 3 point in FP64):
// the tensors go through LDS in whole 16-byte streams, in place; a thread reading and writing its own
// 72-byte record took 315 us for 8.0 M points in FP64, 229 us this way (5.3 TB/s).  In FP32 the two are level
// by themselves (103 and 113 us), but the streaming stores leave the caches to the next kernel: the whole
// force evaluation is 1.5 to 2 % faster.
template <class T, int TD>
__global__ void __launch_bounds__(BS) k_elastic_stress(int64_t n, const T* __restrict__ eps, const T* __restrict__ K,
                                                       const T* __restrict__ G, T* __restrict__ sig)
{
    __shared__ __align__(16) T s_t[BS * TD * TD];
    const int64_t p0 = blockIdx.x * static_cast<int64_t>(BS);
    const int np = static_cast<int>(min<int64_t>(BS, n - p0));
    const int64_t p = p0 + min(static_cast<int>(threadIdx.x), np - 1);
    const T k = K[p], g = G[p];
    stage_in<T, BS, (TD * TD * sizeof(T) + 15) / 16>(s_t, eps + p0 * TD * TD, np * TD * TD);
    __syncthreads();
    if (threadIdx.x < np) {
        T* s = s_t + threadIdx.x * TD * TD;
        T e[TD * TD];
#pragma unroll
        for (int i = 0; i < TD * TD; ++i) e[i] = s[i];
        T tr = (TD == 3) ? e[0] + e[4] + e[8] : e[0] + e[3];
#pragma unroll
        for (int i = 0; i < TD; ++i)
#pragma unroll
            for (int j = 0; j < TD; ++j) {
                if (i == j) s[i * TD + j] = k * tr + T(2) * g * (e[i * TD + j] - tr / T(3));
                else s[i * TD + j] = T(2) * g * e[i * TD + j];
            }
    }
    __syncthreads();
    stage_out<T, BS>(sig + p0 * TD * TD, s_t, np * TD * TD);
}

// Tangent C_ijab = K d_ij d_ab + 2 G (0.5 (d_ia d_jb + d_ib d_ja) - d_ij d_ab / 3) per point.  Every
// point has four distinct entries: K + 2G (1 - 1/3) (i = j = a = b), K + 2G (-1/3) (i = j, a = b,
// i != a), G ({a, b} = {i, j}, i != j) and 0, each formed from the same FP64 expression as the
// per-point loop of the material law (TO = float rounds it once).  A workgroup computes the four
// entries of its TP points into LDS, then writes its contiguous slice of C with full-wave
// contiguous 16-byte streaming stores: GP points (GP TD^4 entries) are NV stores, and a small LDS
// table gives, for each store of a group, the point and entry of each of its ES lanes.
constexpr int TP = 256;

// entry code of component c = ((i TD + j) TD + a) TD + b
template <int TD>
__device__ inline int tangent_code(int c)
{
    const int i = c / (TD * TD * TD), j = (c / (TD * TD)) % TD, a = (c / TD) % TD, b = c % TD;
    if (i == j && a == b) return i == a ? 0 : 1;
    if (i != j && ((i == a && j == b) || (i == b && j == a))) return 2;
    return 3;
}

template <int TD, class TO>
__global__ void __launch_bounds__(BS) k_elastic_tangent(int64_t n, const double* __restrict__ K,
                                                        const double* __restrict__ G, TO* __restrict__ C, bool vec)
{
    static_assert(BS == TP, "one point per thread in the first phase");
    constexpr int T4 = TD * TD * TD * TD;
    constexpr int ES = 16 / static_cast<int>(sizeof(TO));  // entries per 16-byte store
    constexpr int GP = T4 % ES == 0 ? 1 : ES;               // points per group (GP T4 a multiple of ES)
    constexpr int NV = GP * T4 / ES;                        // stores per group
    constexpr int NS = TP / GP * NV;                        // stores per workgroup
    typedef TO V __attribute__((ext_vector_type(ES)));
    __shared__ TO s_val[TP][4];
    __shared__ uint16_t s_tab[NV];
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * TP;
    const int np = static_cast<int>(min<int64_t>(TP, n - p0));
    if (threadIdx.x < np) {
        const double k = K[p0 + threadIdx.x], g = G[p0 + threadIdx.x];
        const double a2_0 = 0.5 * (1.0 * 1.0 + 1.0 * 1.0) - 1.0 * 1.0 / 3.0; // i = j = a = b
        const double a2_1 = 0.5 * (0.0 * 0.0 + 0.0 * 0.0) - 1.0 * 1.0 / 3.0; // i = j != a = b
        s_val[threadIdx.x][0] = static_cast<TO>(k * 1.0 * 1.0 + 2.0 * g * a2_0);
        s_val[threadIdx.x][1] = static_cast<TO>(k * 1.0 * 1.0 + 2.0 * g * a2_1);
        s_val[threadIdx.x][2] = static_cast<TO>(k * 0.0 * 0.0 + 2.0 * g * (0.5 * (1.0 * 1.0 + 0.0 * 0.0) - 0.0 * 0.0 / 3.0));
        s_val[threadIdx.x][3] = static_cast<TO>(k * 0.0 * 0.0 + 2.0 * g * (0.5 * (0.0 * 0.0 + 0.0 * 0.0) - 0.0 * 0.0 / 3.0));
    }
    for (int v = threadIdx.x; v < NV; v += BS) {
        uint16_t t = 0;
#pragma unroll
        for (int l = 0; l < ES; ++l) {
            const int f = v * ES + l, off = f / T4;
            t |= static_cast<uint16_t>((off | (tangent_code<TD>(f - off * T4) << 2)) << (4 * l));
        }
        s_tab[v] = t;
    }
    __syncthreads();
    TO* out = C + p0 * T4;
    if (vec && np == TP) {
        V* o = reinterpret_cast<V*>(out);
        for (int sidx = threadIdx.x; sidx < NS; sidx += BS) {
            const int grp = sidx / NV, v = sidx - grp * NV;
            const unsigned t = s_tab[v];
            V w;
#pragma unroll
            for (int l = 0; l < ES; ++l) {
                const unsigned e = (t >> (4 * l)) & 15u;
                w[l] = s_val[grp * GP + (e & 3u)][e >> 2];
            }
            __builtin_nontemporal_store(w, o + sidx);
        }
    }
    else {
        for (int f = threadIdx.x; f < np * T4; f += BS) {
            const int pl = f / T4;
            out[f] = s_val[pl][tangent_code<TD>(f - pl * T4)];
        }
    }
}

void compute_geometry(gf_quad_s* q, hipStream_t s)
{
    int64_t n = q->nelem * q->nip;
    if (n == 0) return;
    if (q->et == GF_HEX8)
        k_compute_dN_hex8<<<nblocks(n, BS), BS, 0, s>>>(n, q->nip, q->x.p, q->dNxi_d.p, q->w_d.p, q->dNx.p, q->vol.p);
    else
        k_compute_dN_quad4<<<nblocks(n, BS), BS, 0, s>>>(n, q->nip, q->et == GF_QUAD4_PLANAR, q->thick, q->x.p,
                                                       q->dNxi_d.p, q->w_d.p, q->dNx.p, q->vol.p);
    check_launch();
    q->have32 = false;
}

void ensure32(gf_quad_s* q, hipStream_t s)
{
    if (q->have32) return;
    int64_t n1 = q->nelem * q->nip * q->nne * q->ndim, n2 = q->nelem * q->nip;
    if (q->dNx32.n != static_cast<size_t>(n1)) q->dNx32.alloc(n1);
    if (q->vol32.n != static_cast<size_t>(n2)) q->vol32.alloc(n2);
    if (n2 && q->et == GF_HEX8 && geo32_lds_bytes(q->nip) <= 65536)
        k_geometry32_hex8<<<nblocks(n2, GB32), GB32, geo32_lds_bytes(q->nip), s>>>(n2, q->nip, q->x.p, q->dNxi_d.p,
                                                                                  q->w_d.p, q->dNx32.p, q->vol32.p);
    else if (n2) {
        k_to_f32<<<nblocks(n1, BS), BS, 0, s>>>(n1, q->dNx.p, q->dNx32.p);
        k_to_f32<<<nblocks(n2, BS), BS, 0, s>>>(n2, q->vol.p, q->vol32.p);
    }
    check_launch();
    q->have32 = true;
}

int grad_dispatch(gf_quad q, const void* elemvec, void* qtensor, int dtype, int mode, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && elemvec && qtensor, "null argument");
        GF_REQUIRE(dtype == GF_F64 || dtype == GF_F32, "dtype must be GF_F64 or GF_F32");
        int64_t n = q->nelem * q->nip;
        if (n == 0) return;
        hipStream_t s = S(stream);
        auto geometry = [&](auto tag) { // the stored dN/dx in the arithmetic's type
            if constexpr (std::is_same_v<decltype(tag), float>) {
                ensure32(q, s);
                return static_cast<const float*>(q->dNx32.p);
            }
            else
                return static_cast<const double*>(q->dNx.p);
        };
        auto launch = [&](auto tag, auto mtag, const auto* u, auto* o) {
            using T = decltype(tag);
            constexpr int M = decltype(mtag)::value;
            const size_t sz = sizeof(T);
            // the geometry is recomputed from the coordinates, except for Hex8 in FP32, where the FP64
            // recomputation (some 430 FP64 operations per point) takes as long as 768 bytes per element
            // of stored FP32 geometry do (395 k elements: 85 against 80 us), and a Hex8 rule of one
            // point, whose workgroups span too many elements for LDS
            if (q->et == GF_HEX8) {
                if constexpr (std::is_same_v<T, double>) {
                    if (grad3x_lds_bytes(q->nip, sz) <= 65536) {
                        k_grad_3d_x<T, M><<<nblocks(n, QB3), QB3, grad3x_lds_bytes(q->nip, sz), s>>>(
                            n, q->nip, q->x.p, q->dNxi_d.p, u, o);
                        return;
                    }
                }
                k_grad_3d_lds<T, M><<<nblocks(n, 128), 128, grad3_lds_bytes(128, q->nip, sz), s>>>(
                    n, q->nip, geometry(tag), u, o);
            }
            else if (q->et == GF_QUAD4_PLANAR)
                k_grad_2d_x<T, 3, M><<<nblocks(n, 256), 256, grad2x_lds_bytes(q->nip, 3, sz), s>>>(n, q->nip, q->x.p,
                                                                                                   q->dNxi_d.p, u, o);
            else
                k_grad_2d_x<T, 2, M><<<nblocks(n, 256), 256, grad2x_lds_bytes(q->nip, 2, sz), s>>>(n, q->nip, q->x.p,
                                                                                                   q->dNxi_d.p, u, o);
        };
        auto by_mode = [&](auto tag, const auto* u, auto* o) {
            if (mode == 0) launch(tag, std::integral_constant<int, 0>(), u, o);
            else if (mode == 1) launch(tag, std::integral_constant<int, 1>(), u, o);
            else launch(tag, std::integral_constant<int, 2>(), u, o);
        };
        if (dtype == GF_F64) by_mode(double(0), static_cast<const double*>(elemvec), static_cast<double*>(qtensor));
        else by_mode(float(0), static_cast<const float*>(elemvec), static_cast<float*>(qtensor));
        check_launch();
    });
}

} // namespace

// Accessors used by other translation units (stiffness, explicit).
namespace gf {
const double* quad_dNx(gf_quad q) { return q->dNx.p; }
const double* quad_vol(gf_quad q) { return q->vol.p; }
int quad_etype(gf_quad q) { return q->et; }
int64_t quad_nelem(gf_quad q) { return q->nelem; }
int quad_nip(gf_quad q) { return q->nip; }
uint64_t quad_version(gf_quad q) { return q->version; }
} // namespace gf

extern "C" {

int gf_quad_create(gf_quad* out, int etype, const double* x, int64_t nelem, int rule, const double* xi_h,
                   const double* w_h, int nip, double thick, void* stream)
{
    return guard([&] {
        GF_REQUIRE(out && x, "null argument");
        GF_REQUIRE(etype == GF_QUAD4 || etype == GF_QUAD4_PLANAR || etype == GF_HEX8, "unknown element type");
        auto q = new gf_quad_s();
        try {
            q->et = etype;
            q->nne = etype == GF_HEX8 ? 8 : 4;
            q->ndim = etype == GF_HEX8 ? 3 : 2;
            q->tdim = etype == GF_QUAD4 ? 2 : 3;
            q->nelem = nelem;
            q->thick = thick;
            if (xi_h && w_h) {
                GF_REQUIRE(nip > 0, "nip > 0 with a custom rule");
                q->xi.assign(xi_h, xi_h + nip * q->ndim);
                q->w.assign(w_h, w_h + nip);
            }
            else {
                GF_REQUIRE(rule == GF_GAUSS || rule == GF_NODAL, "rule must be GF_GAUSS or GF_NODAL");
                default_rule(etype, rule, q->xi, q->w);
            }
            q->nip = static_cast<int>(q->w.size());
            q->N.resize(q->nip * q->nne);
            q->dNxi.resize(q->nip * q->nne * q->ndim);
            shape_functions(etype, q->nip, q->xi.data(), q->N.data(), q->dNxi.data());
            q->N_d.upload(q->N);
            q->dNxi_d.upload(q->dNxi);
            q->w_d.upload(q->w);
            q->x.alloc(nelem * q->nne * q->ndim);
            if (q->x.n)
                GF_HIP(hipMemcpyAsync(q->x.p, x, q->x.n * sizeof(double), hipMemcpyDeviceToDevice, S(stream)));
            q->dNx.alloc(nelem * q->nip * q->nne * q->ndim);
            q->vol.alloc(nelem * q->nip);
            compute_geometry(q, S(stream));
        }
        catch (...) {
            delete q;
            throw;
        }
        *out = q;
    });
}

int gf_quad_destroy(gf_quad q)
{
    delete q;
    return GF_OK;
}

int gf_quad_sizes(gf_quad q, int64_t* nelem, int* nne, int* ndim, int* tdim, int* nip)
{
    return guard([&] {
        GF_REQUIRE(q, "null quadrature");
        if (nelem) *nelem = q->nelem;
        if (nne) *nne = q->nne;
        if (ndim) *ndim = q->ndim;
        if (tdim) *tdim = q->tdim;
        if (nip) *nip = q->nip;
    });
}

int gf_quad_update_x(gf_quad q, const double* x, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && x, "null argument");
        ++q->version;
        if (q->x.n)
            GF_HIP(hipMemcpyAsync(q->x.p, x, q->x.n * sizeof(double), hipMemcpyDeviceToDevice, S(stream)));
        compute_geometry(q, S(stream));
    });
}

int gf_quad_gradN(gf_quad q, const double** dNx)
{
    return guard([&] {
        GF_REQUIRE(q && dNx, "null argument");
        *dNx = q->dNx.p;
    });
}

int gf_quad_dV(gf_quad q, const double** dV)
{
    return guard([&] {
        GF_REQUIRE(q && dV, "null argument");
        *dV = q->vol.p;
    });
}

int gf_quad_interp_quad_vector(gf_quad q, const double* elemvec, int nv, double* qvector, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && elemvec && qvector && nv > 0, "invalid argument");
        int64_t n = q->nelem * q->nip;
        if (n == 0) return;
        k_interp<<<nblocks(n, BS), BS, 0, S(stream)>>>(n, q->nip, q->nne, nv, q->N_d.p, elemvec, qvector);
        check_launch();
    });
}

int gf_quad_gradN_vector(gf_quad q, const void* elemvec, void* qtensor, int dtype, void* stream)
{
    return grad_dispatch(q, elemvec, qtensor, dtype, 0, stream);
}

int gf_quad_gradN_vector_T(gf_quad q, const void* elemvec, void* qtensor, int dtype, void* stream)
{
    return grad_dispatch(q, elemvec, qtensor, dtype, 1, stream);
}

int gf_quad_symgradN_vector(gf_quad q, const void* elemvec, void* qtensor, int dtype, void* stream)
{
    return grad_dispatch(q, elemvec, qtensor, dtype, 2, stream);
}

int gf_quad_int_N_vector_dV(gf_quad q, const double* qvector, int nv, double* elemvec, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && qvector && elemvec && nv > 0, "invalid argument");
        int64_t n = q->nelem * q->nne;
        if (n == 0) return;
        k_int_N_vector<<<nblocks(n, BS), BS, 0, S(stream)>>>(n, q->nip, q->nne, nv, q->N_d.p, q->vol.p, qvector,
                                                           elemvec);
        check_launch();
    });
}

int gf_quad_int_N_scalar_NT_dV(gf_quad q, const double* qscalar, double* elemmat, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && qscalar && elemmat, "null argument");
        int64_t n = q->nelem * q->nne * q->nne;
        if (n == 0) return;
        k_int_N_scalar<<<nblocks(n, BS), BS, 0, S(stream)>>>(n, q->nip, q->nne, q->ndim, q->N_d.p, q->vol.p, qscalar,
                                                           elemmat);
        check_launch();
    });
}

int gf_quad_int_gradN_dot_tensor2_dV(gf_quad q, const void* qtensor, void* elemvec, int dtype, void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && qtensor && elemvec, "null argument");
        GF_REQUIRE(dtype == GF_F64 || dtype == GF_F32, "dtype must be GF_F64 or GF_F32");
        const int64_t E = q->nelem;
        if (E == 0) return;
        hipStream_t s = S(stream);
        auto launch = [&](auto tag, const auto* in, auto* o) {
            using T = decltype(tag);
            const size_t sz = sizeof(T);
            const int nip = q->nip;
            // rules of more points than a workgroup has threads, or whose points' LDS outgrows 64 KiB: the
            // unstaged kernel with the stored geometry, thread per (e, m)
            const bool staged = q->et == GF_HEX8 ? nip <= PB3 && int2_h8_lds_bytes(nip, sz) <= 65536
                                                 : nip <= PB2 && int2_q4_lds_bytes(nip, 3, sz) <= 65536;
            if (!staged) {
                const T *g, *v;
                if constexpr (std::is_same_v<T, float>) {
                    ensure32(q, s);
                    g = q->dNx32.p;
                    v = q->vol32.p;
                }
                else {
                    g = q->dNx.p;
                    v = q->vol.p;
                }
                const int64_t n = E * q->nne;
                if (q->et == GF_HEX8) k_int_tensor2<T, 3, 3><<<nblocks(n, BS), BS, 0, s>>>(n, nip, q->nne, g, v, in, o);
                else if (q->et == GF_QUAD4_PLANAR)
                    k_int_tensor2<T, 2, 3><<<nblocks(n, BS), BS, 0, s>>>(n, nip, q->nne, g, v, in, o);
                else k_int_tensor2<T, 2, 2><<<nblocks(n, BS), BS, 0, s>>>(n, nip, q->nne, g, v, in, o);
                return;
            }
            if (q->et == GF_HEX8) {
                const T *gx, *gv;
                if constexpr (std::is_same_v<T, float>) {
                    ensure32(q, s);
                    gx = q->dNx32.p;
                    gv = q->vol32.p;
                }
                else {
                    gx = q->x.p;
                    gv = q->w_d.p;
                }
                if constexpr (std::is_same_v<T, float>) {
                    if (E >= H8_STAGED && int2_h8_staged_lds_bytes(nip) <= 32768) {
                        k_int_tensor2_h8_staged<<<nblocks(E, EBS), EBS * 8, int2_h8_staged_lds_bytes(nip), s>>>(E, nip, gx, gv,
                                                                                                               in, o);
                        return;
                    }
                }
                k_int_tensor2_h8<T><<<nblocks(E, PB3 / nip), PB3, int2_h8_lds_bytes(nip, sz), s>>>(
                    E, nip, gx, q->dNxi_d.p, gv, in, o);
            }
            else if (q->et == GF_QUAD4_PLANAR)
                k_int_tensor2_q4<T, 3><<<nblocks(E, PB2 / nip), PB2, int2_q4_lds_bytes(nip, 3, sz), s>>>(
                    E, nip, 1, q->thick, q->x.p, q->dNxi_d.p, q->w_d.p, in, o);
            else
                k_int_tensor2_q4<T, 2><<<nblocks(E, PB2 / nip), PB2, int2_q4_lds_bytes(nip, 2, sz), s>>>(
                    E, nip, 0, q->thick, q->x.p, q->dNxi_d.p, q->w_d.p, in, o);
        };
        if (dtype == GF_F64) launch(double(0), static_cast<const double*>(qtensor), static_cast<double*>(elemvec));
        else launch(float(0), static_cast<const float*>(qtensor), static_cast<float*>(elemvec));
        check_launch();
    });
}

int gf_quad_int_gradN_dot_tensor4_dot_gradNT_dV(gf_quad q, const double* C, double* elemmat, int precision,
                                                void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && C && elemmat, "null argument");
        int64_t n = q->nelem * q->nne * q->nne;
        if (n == 0) return;
        hipStream_t s = S(stream);
        if (precision == GF_BF16X3) {
            GF_REQUIRE(q->et == GF_HEX8, "GF_BF16X3 is implemented for Hex8");
            int rc = gf::stiffness_bf16x3(q, C, elemmat, s);
            if (rc != GF_OK) throw Error(rc, gf_last_error());
            return;
        }
        GF_REQUIRE(precision == GF_F64, "precision must be GF_F64 or GF_BF16X3");
        if (q->et == GF_HEX8 && q->nip == 8) {
            int rc = gf::stiffness_f64_hex8(q, C, elemmat, s);
            if (rc != GF_OK) throw Error(rc, gf_last_error());
            return;
        }
        if (q->et != GF_HEX8 && q->nip == 4 && aligned16(elemmat)) {
            if (q->et == GF_QUAD4_PLANAR)
                k_int_tensor4_q4_f64<3><<<nblocks(q->nelem, T4_EB), 4 * T4_EB, 0, s>>>(q->nelem, q->dNx.p, q->vol.p, C,
                                                                                        elemmat);
            else
                k_int_tensor4_q4_f64<2><<<nblocks(q->nelem, T4_EB), 4 * T4_EB, 0, s>>>(q->nelem, q->dNx.p, q->vol.p, C,
                                                                                        elemmat);
        }
        else if (q->et == GF_HEX8)
            k_int_tensor4_f64<8, 3, 3><<<nblocks(n, BS), BS, 0, s>>>(n, q->nip, q->dNx.p, q->vol.p, C, elemmat);
        else if (q->et == GF_QUAD4_PLANAR)
            k_int_tensor4_f64<4, 2, 3><<<nblocks(n, BS), BS, 0, s>>>(n, q->nip, q->dNx.p, q->vol.p, C, elemmat);
        else
            k_int_tensor4_f64<4, 2, 2><<<nblocks(n, BS), BS, 0, s>>>(n, q->nip, q->dNx.p, q->vol.p, C, elemmat);
        check_launch();
    });
}

int gf_material_elastic_stress(int64_t nq, int tdim, const void* eps, const void* K, const void* G, void* sig,
                               int dtype, void* stream)
{
    return guard([&] {
        GF_REQUIRE(eps && K && G && sig, "null argument");
        GF_REQUIRE(tdim == 2 || tdim == 3, "tdim must be 2 or 3");
        GF_REQUIRE(dtype == GF_F64 || dtype == GF_F32, "dtype must be GF_F64 or GF_F32");
        if (nq == 0) return;
        hipStream_t s = S(stream);
        unsigned nb = nblocks(nq, BS);
        if (dtype == GF_F64) {
            auto e = static_cast<const double*>(eps);
            auto k = static_cast<const double*>(K);
            auto g = static_cast<const double*>(G);
            auto o = static_cast<double*>(sig);
            if (tdim == 3) k_elastic_stress<double, 3><<<nb, BS, 0, s>>>(nq, e, k, g, o);
            else k_elastic_stress<double, 2><<<nb, BS, 0, s>>>(nq, e, k, g, o);
        }
        else {
            auto e = static_cast<const float*>(eps);
            auto k = static_cast<const float*>(K);
            auto g = static_cast<const float*>(G);
            auto o = static_cast<float*>(sig);
            if (tdim == 3) k_elastic_stress<float, 3><<<nb, BS, 0, s>>>(nq, e, k, g, o);
            else k_elastic_stress<float, 2><<<nb, BS, 0, s>>>(nq, e, k, g, o);
        }
        check_launch();
    });
}

int gf_material_elastic_tangent(int64_t nq, int tdim, const double* K, const double* G, double* C, void* stream)
{
    return guard([&] {
        GF_REQUIRE(K && G && C, "null argument");
        GF_REQUIRE(tdim == 2 || tdim == 3, "tdim must be 2 or 3");
        if (nq == 0) return;
        if (tdim == 3) k_elastic_tangent<3, double><<<nblocks(nq, TP), BS, 0, S(stream)>>>(nq, K, G, C, aligned16(C));
        else k_elastic_tangent<2, double><<<nblocks(nq, TP), BS, 0, S(stream)>>>(nq, K, G, C, aligned16(C));
        check_launch();
    });
}

int gf_material_elastic_tangent_f32(int64_t nq, int tdim, const double* K, const double* G, float* C, void* stream)
{
    return guard([&] {
        GF_REQUIRE(K && G && C, "null argument");
        GF_REQUIRE(tdim == 2 || tdim == 3, "tdim must be 2 or 3");
        if (nq == 0) return;
        if (tdim == 3) k_elastic_tangent<3, float><<<nblocks(nq, TP), BS, 0, S(stream)>>>(nq, K, G, C, aligned16(C));
        else k_elastic_tangent<2, float><<<nblocks(nq, TP), BS, 0, S(stream)>>>(nq, K, G, C, aligned16(C));
        check_launch();
    });
}

} // extern "C"
