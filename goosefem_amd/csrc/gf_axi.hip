// Element::Quad4::QuadratureAxisymmetric (include/GooseFEM/ElementQuad4Axisymmetric.h:33-467) on the
// device.  Nodal coordinates are (z, r); tensors are in (r, theta, z) order.  Of the reference's
// B-matrix [nelem, nip, nne, 3, 3, 3] only five components per node are non-zero (:401-438):
//   B(m,r,r,r) = B(m,r,z,z) = dN/dr,  B(m,t,t,r) = N / r_q,  B(m,z,r,r) = B(m,z,z,z) = dN/dz,
// so the geometry is kept as G[e, q, m] = (dN/dr, N / r_q, dN/dz) (12 doubles per point instead of
// 108) and dV = w J 2 pi r_q; the kernels that are bound by HBM form it again from the element's 64 bytes
// of coordinates, with the function that made the stored one.  Every kernel keeps the reference's FP64
// expression and summation order (no contraction), so results equal the reference's bit for bit.  The
// stiffness runs the 25 products of each node pair over the five non-zero slots a (outer) and b (inner), slot =
// (i, j, value, nodal component): (r,r: dN/dr, u_r) (t,t: N/r, u_r) (z,z: dN/dz, u_z)
// (r,z: dN/dr, u_z) (z,r: dN/dz, u_r), and K(m, c_a; n, c_b) += B_a(m) C(i_a, j_a, j_b, i_b) B_b(n) dV
// (:298-398, in the listed order).
#include "gf_internal.hpp"
#include "gf_stage.hpp"

using namespace gf;

namespace {

constexpr int MAXQ = 16;

struct AxiRule {
    int nip;
    double N[MAXQ][4], dNxi[MAXQ][4][2], w[MAXQ];
};

} // namespace

struct gf_axi_s {
    int64_t nelem = 0;
    AxiRule rule;
    DBuf<double> x, G, vol;
};

namespace {

constexpr int BS = 256;

// G (12) and dV of point q of the element with coordinates xv
__device__ inline void axi_point_geometry(const AxiRule& R, int q, const double* __restrict__ xv, double* o, double& v)
{
    const double(*g)[2] = R.dNxi[q];
    const double* n = R.N[q];
    const double J00 = g[0][0] * xv[0] + g[1][0] * xv[2] + g[2][0] * xv[4] + g[3][0] * xv[6];
    const double J01 = g[0][0] * xv[1] + g[1][0] * xv[3] + g[2][0] * xv[5] + g[3][0] * xv[7];
    const double J10 = g[0][1] * xv[0] + g[1][1] * xv[2] + g[2][1] * xv[4] + g[3][1] * xv[6];
    const double J11 = g[0][1] * xv[1] + g[1][1] * xv[3] + g[2][1] * xv[5] + g[3][1] * xv[7];
    // cofactor inverse (include/GooseFEM/detail.h:17-70)
    const double det = J00 * J11 - J01 * J10;
    const double I00 = J11 / det, I01 = -1.0 * J01 / det, I10 = -1.0 * J10 / det, I11 = J00 / det;
    const double rq = n[0] * xv[1] + n[1] * xv[3] + n[2] * xv[5] + n[3] * xv[7];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        o[3 * m + 0] = I10 * g[m][0] + I11 * g[m][1];
        o[3 * m + 1] = 1.0 / rq * n[m];
        o[3 * m + 2] = I00 * g[m][0] + I01 * g[m][1];
    }
    v = R.w[q] * det * 2.0 * M_PI * rq;
}

__global__ void k_axi_geometry(int64_t nelem, AxiRule R, const double* __restrict__ x, double* __restrict__ G,
                               double* __restrict__ vol)
{
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= nelem * R.nip) return;
    const int64_t e = t / R.nip;
    const int q = static_cast<int>(t - e * R.nip);
    axi_point_geometry(R, q, x + 8 * e, G + 12 * t, vol[t]);
}

// gradN_vector (mode 0, :140-169), gradN_vector_T (1, :171-200), symGradN_vector (2, :202-233).
// A workgroup owns BS / nip whole elements, one thread per point; coordinates, element vectors and tensors
// go through LDS as contiguous 16-byte streams.  Bound by HBM, 416 bytes per element (736 with the stored
// geometry): 300 k elements 47 -> 24.5 us.
__global__ void __launch_bounds__(BS) k_axi_grad(int64_t nelem, AxiRule R, int mode, const double* __restrict__ x,
                                                 const double* __restrict__ u_, double* __restrict__ out)
{
    extern __shared__ __align__(16) double smem[];
    const int EB = BS / R.nip;
    double *s_o = smem, *s_x = s_o + 9 * BS, *s_u = s_x + 8 * EB;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * EB;
    const int ne = static_cast<int>(min<int64_t>(EB, nelem - e0)), np = ne * R.nip;
    stage_in<double, BS, 1>(s_x, x + 8 * e0, 8 * ne);
    stage_in<double, BS, 1>(s_u, u_ + 8 * e0, 8 * ne);
    __syncthreads();
    if (threadIdx.x < np) {
        const int el = threadIdx.x / R.nip, q = threadIdx.x - el * R.nip;
        double b[12], v;
        axi_point_geometry(R, q, s_x + 8 * el, b, v);
        const double* u = s_u + 8 * el; // (u_z, u_r) per node
        const double rr = b[0] * u[1] + b[3] * u[3] + b[6] * u[5] + b[9] * u[7];
        const double tt = b[1] * u[1] + b[4] * u[3] + b[7] * u[5] + b[10] * u[7];
        const double zz = b[2] * u[0] + b[5] * u[2] + b[8] * u[4] + b[11] * u[6];
        double r2, r6;
        if (mode == 2) {
            r2 = r6 = 0.5 * (b[0] * u[0] + b[3] * u[2] + b[6] * u[4] + b[9] * u[6] + b[2] * u[1] + b[5] * u[3] +
                             b[8] * u[5] + b[11] * u[7]);
        }
        else {
            const double dzr = b[0] * u[0] + b[3] * u[2] + b[6] * u[4] + b[9] * u[6];
            const double drz = b[2] * u[1] + b[5] * u[3] + b[8] * u[5] + b[11] * u[7];
            r2 = mode == 0 ? dzr : drz;
            r6 = mode == 0 ? drz : dzr;
        }
        double* o = s_o + 9 * threadIdx.x;
        o[0] = rr;
        o[1] = 0.0;
        o[2] = r2;
        o[3] = 0.0;
        o[4] = tt;
        o[5] = 0.0;
        o[6] = r6;
        o[7] = 0.0;
        o[8] = zz;
    }
    __syncthreads();
    stage_out<double, BS>(out + 9 * e0 * R.nip, s_o, 9 * np);
}

// int_N_scalar_NT_dV (:235-266)
__global__ void k_axi_int_N(int64_t nelem, AxiRule R, const double* __restrict__ vol, const double* __restrict__ qs,
                            double* __restrict__ M)
{
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= nelem * 16) return;
    const int64_t e = t / 16;
    const int m = static_cast<int>(t % 16) / 4, k = static_cast<int>(t % 4);
    double a = 0.0, c = 0.0;
    for (int q = 0; q < R.nip; ++q) {
        const double v = vol[e * R.nip + q], rho = qs[e * R.nip + q];
        a += R.N[q][m] * rho * R.N[q][k] * v;
        c += R.N[q][m] * rho * R.N[q][k] * v;
    }
    double* Me = M + 64 * e;
    Me[(2 * m) * 8 + 2 * k] = a;
    Me[(2 * m) * 8 + 2 * k + 1] = 0.0;
    Me[(2 * m + 1) * 8 + 2 * k] = 0.0;
    Me[(2 * m + 1) * 8 + 2 * k + 1] = c;
}

// int_gradN_dot_tensor2_dV (:268-296): one thread per point forms the point's contributions to the four
// nodes (in place of its tensor in LDS), then one thread per (element, node) adds them in point order.
// Bound by HBM, 416 bytes per element (768 with the stored geometry): 300 k elements
// 47.5 -> 26 us.
__global__ void __launch_bounds__(BS) k_axi_int_t2(int64_t nelem, AxiRule R, const double* __restrict__ x,
                                                   const double* __restrict__ sig, double* __restrict__ f)
{
    extern __shared__ __align__(16) double smem[];
    const int EB = BS / R.nip;
    double *s_s = smem, *s_x = s_s + 9 * BS; // s_x: coordinates, then the element vectors
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * EB;
    const int ne = static_cast<int>(min<int64_t>(EB, nelem - e0)), np = ne * R.nip;
    stage_in<double, BS, 5>(s_s, sig + 9 * e0 * R.nip, 9 * np);
    stage_in<double, BS, 1>(s_x, x + 8 * e0, 8 * ne);
    __syncthreads();
    if (threadIdx.x < np) {
        const int el = threadIdx.x / R.nip, q = threadIdx.x - el * R.nip;
        double b[12], v, s[9];
        axi_point_geometry(R, q, s_x + 8 * el, b, v);
        double* c = s_s + 9 * threadIdx.x;
#pragma unroll
        for (int k = 0; k < 9; ++k) s[k] = c[k];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            c[2 * m] = v * (b[3 * m + 2] * s[8] + b[3 * m] * s[2]);
            c[2 * m + 1] = v * (b[3 * m] * s[0] + b[3 * m + 1] * s[4] + b[3 * m + 2] * s[6]);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 4 * ne; t += BS) {
        const double* c = s_s + (t / 4) * R.nip * 9 + 2 * (t % 4);
        double f0 = 0.0, f1 = 0.0;
        for (int q = 0; q < R.nip; ++q) {
            f0 += c[9 * q];
            f1 += c[9 * q + 1];
        }
        s_x[2 * t] = f0;
        s_x[2 * t + 1] = f1;
    }
    __syncthreads();
    stage_out<double, BS>(f + 8 * e0, s_x, 8 * ne);
}

// int_gradN_dot_tensor4_dot_gradNT_dV (:298-398), one thread per (element, node m): per point the products
// B_a(m) C are formed once and used for all four column nodes, in the listed order.  A workgroup owns 64
// elements.  Four points at a time each thread forms the geometry of one of them; the 25 entries of a
// point's tangents go to registers one point ahead and through LDS, and so do the rows of K_e, which leave
// as one 16-byte stream (scalar stores if elemmat is not 16-byte aligned).  Bound by HBM: the tangents (all
// of a 648-byte record's lines hold a used entry) and K_e.  225 k elements: 128 us, 285 us with one
// thread per node pair reading its own tangent and storing its own 2 x 2 block.
constexpr int T4_EB = 64, T4_KROW = 18, T4_NC = (25 * T4_EB + BS - 1) / BS;

__global__ void __launch_bounds__(BS, 4) k_axi_int_t4(int64_t nelem, AxiRule R, const double* __restrict__ x,
                                                   const double* __restrict__ C, double* __restrict__ K)
{
    static_assert(BS == 4 * T4_EB, "one thread per (element, node)");
    constexpr int si[5] = {0, 1, 2, 0, 2}, sj[5] = {0, 1, 2, 2, 0}, sv[5] = {0, 1, 2, 0, 2}, sc[5] = {1, 1, 0, 0, 1};
    typedef double d2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double smem[T4_EB * (4 * 13 + 25)];
    static_assert(T4_EB * (4 * 13 + 25) >= BS * T4_KROW, "the rows of K must fit");
    double *s_g = smem, *s_c = smem + T4_EB * 4 * 13; // [element][point of four][G, dV], [element][25]
    const int t = threadIdx.x, el = t / 4, m = t % 4, nip = R.nip;
    const int64_t e0 = blockIdx.x * static_cast<int64_t>(T4_EB);
    const int ne = static_cast<int>(min<int64_t>(T4_EB, nelem - e0));
    // entry (a, b) of a tangent is its (i_a, j_a, j_b, i_b) component: both pairs at even positions of nine
    const double* Cb = C + e0 * nip * 81;
    int src[T4_NC];
#pragma unroll
    for (int k = 0; k < T4_NC; ++k) {
        const int w = min(t + k * BS, 25 * ne - 1), r = w % 25, a = r / 5, b = r % 5;
        const int ia = a < 3 ? 4 * a : a == 3 ? 2 : 6, jb = b < 3 ? 4 * b : b == 3 ? 6 : 2;
        src[k] = (w / 25) * nip * 81 + 9 * ia + jb;
    }
    double pre[T4_NC];
#pragma unroll
    for (int k = 0; k < T4_NC; ++k) pre[k] = Cb[src[k]];
    double acc[4][2][2] = {};
    for (int q0 = 0; q0 < nip; q0 += 4) {
        if (q0 + m < nip) {
            double o[12], v;
            axi_point_geometry(R, q0 + m, x + 8 * (e0 + min(el, ne - 1)), o, v);
            double* g = s_g + 13 * t;
#pragma unroll
            for (int k = 0; k < 12; ++k) g[k] = o[k];
            g[12] = v;
        }
#pragma unroll 1
        for (int q = q0; q < min(q0 + 4, nip); ++q) {
#pragma unroll
            for (int k = 0; k < T4_NC; ++k)
                if (t + k * BS < 25 * T4_EB) s_c[t + k * BS] = pre[k];
            __syncthreads();
            if (q + 1 < nip) {
#pragma unroll
                for (int k = 0; k < T4_NC; ++k) pre[k] = Cb[src[k] + 81 * (q + 1)];
            }
            const double *g = s_g + 13 * (4 * el + q - q0), *c = s_c + 25 * el;
            const double v = g[12];
            double bn[12], bm[3];
#pragma unroll
            for (int k = 0; k < 12; ++k) bn[k] = g[k];
#pragma unroll
            for (int k = 0; k < 3; ++k) bm[k] = g[3 * m + k];
#pragma unroll
            for (int a = 0; a < 5; ++a)
#pragma unroll
                for (int b = 0; b < 5; ++b) {
                    const double bc = bm[sv[a]] * c[5 * a + b];
#pragma unroll
                    for (int n = 0; n < 4; ++n) acc[n][sc[a]][sc[b]] += bc * bn[3 * n + sv[b]] * v;
                }
            __syncthreads(); // the point's tangents (and, after four, the geometry) are consumed
        }
    }
    {
        d2* row = reinterpret_cast<d2*>(smem + T4_KROW * t); // rows 2 m, 2 m + 1: 16 contiguous doubles
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int n = 0; n < 4; ++n) row[4 * i + n] = d2{acc[n][i][0], acc[n][i][1]};
    }
    __syncthreads();
    double* Kb = K + 64 * e0;
    if ((reinterpret_cast<uintptr_t>(K) & 15) == 0) {
        for (int w = t; w < 32 * ne; w += BS)
            __builtin_nontemporal_store(reinterpret_cast<const d2*>(smem + T4_KROW * (w / 8))[w % 8],
                                        reinterpret_cast<d2*>(Kb) + w);
    }
    else
        for (int w = t; w < 64 * ne; w += BS) Kb[w] = smem[T4_KROW * (w / 16) + w % 16];
}

void compute(gf_axi m, const double* x, hipStream_t s)
{
    const int64_t n = m->nelem * m->rule.nip;
    if (!n) return;
    GF_HIP(hipMemcpyAsync(m->x.p, x, m->x.n * sizeof(double), hipMemcpyDeviceToDevice, s));
    k_axi_geometry<<<nblocks(n, BS), BS, 0, s>>>(m->nelem, m->rule, x, m->G.p, m->vol.p);
    check_launch();
}

} // namespace

extern "C" {

int gf_axi_create(gf_axi* out, int64_t nelem, int nip, const double* x, const double* xi_h, const double* w_h,
                  void* stream)
{
    return guard([&] {
        GF_REQUIRE(out && (x || nelem == 0) && xi_h && w_h, "null argument");
        GF_REQUIRE(nelem >= 0 && nip >= 1 && nip <= MAXQ, "0 <= nelem, 1 <= nip <= 16");
        auto m = new gf_axi_s();
        try {
            m->nelem = nelem;
            AxiRule& R = m->rule;
            R.nip = nip;
            for (int q = 0; q < nip; ++q) {
                const double a = xi_h[2 * q], b = xi_h[2 * q + 1];
                // ElementQuad4Axisymmetric.h:74-96 (the Quad4 shape functions)
                R.N[q][0] = 0.25 * (1.0 - a) * (1.0 - b);
                R.N[q][1] = 0.25 * (1.0 + a) * (1.0 - b);
                R.N[q][2] = 0.25 * (1.0 + a) * (1.0 + b);
                R.N[q][3] = 0.25 * (1.0 - a) * (1.0 + b);
                R.dNxi[q][0][0] = -0.25 * (1.0 - b);
                R.dNxi[q][1][0] = +0.25 * (1.0 - b);
                R.dNxi[q][2][0] = +0.25 * (1.0 + b);
                R.dNxi[q][3][0] = -0.25 * (1.0 + b);
                R.dNxi[q][0][1] = -0.25 * (1.0 - a);
                R.dNxi[q][1][1] = -0.25 * (1.0 + a);
                R.dNxi[q][2][1] = +0.25 * (1.0 + a);
                R.dNxi[q][3][1] = +0.25 * (1.0 - a);
                R.w[q] = w_h[q];
            }
            m->x.alloc(8 * nelem);
            m->G.alloc(12 * nelem * nip);
            m->vol.alloc(nelem * nip);
            compute(m, x, S(stream));
        }
        catch (...) {
            delete m;
            throw;
        }
        *out = m;
    });
}

int gf_axi_destroy(gf_axi m)
{
    delete m;
    return GF_OK;
}

int gf_axi_update_x(gf_axi m, const double* x, void* stream)
{
    return guard([&] {
        GF_REQUIRE(m && (x || m->nelem == 0), "null argument");
        compute(m, x, S(stream));
    });
}

int gf_axi_geometry(gf_axi m, const double** G, const double** dV)
{
    return guard([&] {
        GF_REQUIRE(m, "null argument");
        if (G) *G = m->G.p;
        if (dV) *dV = m->vol.p;
    });
}

int gf_axi_grad(gf_axi m, int mode, const double* elemvec, double* qtensor, void* stream)
{
    return guard([&] {
        GF_REQUIRE(m && elemvec && qtensor, "null argument");
        GF_REQUIRE(mode >= 0 && mode <= 2, "mode: 0 gradN_vector, 1 gradN_vector_T, 2 symGradN_vector");
        if (m->nelem)
            k_axi_grad<<<nblocks(m->nelem, BS / m->rule.nip), BS, (9 * BS + 16 * (BS / m->rule.nip)) * sizeof(double),
                         S(stream)>>>(m->nelem, m->rule, mode, m->x.p, elemvec, qtensor);
        check_launch();
    });
}

int gf_axi_int_N_scalar_NT_dV(gf_axi m, const double* qscalar, double* elemmat, void* stream)
{
    return guard([&] {
        GF_REQUIRE(m && qscalar && elemmat, "null argument");
        if (m->nelem)
            k_axi_int_N<<<nblocks(16 * m->nelem, BS), BS, 0, S(stream)>>>(m->nelem, m->rule, m->vol.p, qscalar, elemmat);
        check_launch();
    });
}

int gf_axi_int_gradN_dot_tensor2_dV(gf_axi m, const double* qtensor, double* elemvec, void* stream)
{
    return guard([&] {
        GF_REQUIRE(m && qtensor && elemvec, "null argument");
        if (m->nelem)
            k_axi_int_t2<<<nblocks(m->nelem, BS / m->rule.nip), BS, (9 * BS + 8 * (BS / m->rule.nip)) * sizeof(double),
                           S(stream)>>>(m->nelem, m->rule, m->x.p, qtensor, elemvec);
        check_launch();
    });
}

int gf_axi_int_gradN_dot_tensor4_dot_gradNT_dV(gf_axi m, const double* qtensor, double* elemmat, void* stream)
{
    return guard([&] {
        GF_REQUIRE(m && qtensor && elemmat, "null argument");
        if (m->nelem)
            k_axi_int_t4<<<nblocks(m->nelem, T4_EB), BS, 0, S(stream)>>>(m->nelem, m->rule, m->x.p, qtensor, elemmat);
        check_launch();
    });
}

} // extern "C"
