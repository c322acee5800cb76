// Hex8 element stiffness Int_gradN_dot_tensor4_dot_gradNT_dV (include/GooseFEM/Element.h:1131-1176):
//   K(m*3+j, n*3+k) = sum_q sum_{i,l} dNx(q,m,i) C_q(i,j,k,l) dNx(q,n,l) dV_q
//
// GF_BF16X3 (matrix cores).  Write kk = (q, j2, i) (72 values) and
//   T[kk][(n,k)] = dV_q sum_l C_q(i, j2, k, l) dNx(q,n,l)                      (72 x 24, VALU, FP32)
//   A[(m,j)][kk] = delta(j, j2) dNx(q,m,i)                                    (24 x 72)
// so that K = A T: one 24 x 72 by 72 x 24 product per element, evaluated on
// v_mfma_f32_32x32x16_bf16 (tile padded to 32 x 32, contraction to 80).  Both operands are split
// x = hi + lo with hi = bf16(x), lo = bf16(x - hi); the product accumulates hi*hi + hi*lo + lo*hi
// in FP32 (the dropped lo*lo term and the bf16 rounding of lo are ~2^-16 relative).
// One wavefront owns one element: C_q (8 x 81) and dNx, dV go through LDS, dNx split into its parts on the
// way; each MFMA lane evaluates the T entries it feeds, the 15 MFMAs accumulate the 32 x 32 tile, and the
// 24 x 24 result leaves through LDS as one contiguous stream.
//
// GF_F64: the same per-entry accumulation order as the reference loop (q, i, l for each (j, k)) on the
// vector units, four elements per wavefront (k_stiffness_f64).
#include <type_traits>

#include "gf_internal.hpp"

using namespace gf;

namespace gf {
const double* quad_dNx(gf_quad q);
const double* quad_vol(gf_quad q);
int64_t quad_nelem(gf_quad q);
int quad_nip(gf_quad q);
int quad_etype(gf_quad q);
} // namespace gf

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int WAVES = 4;           // wavefronts per workgroup
constexpr int NQ = 8, NN = 8;      // quadrature points, nodes
constexpr int NC = NQ * 81;        // tensor4 doubles per element
constexpr int NG = NQ * NN * 3;    // dNx doubles per element
constexpr int KKP = 80;            // contraction length 72, padded to 5 x 16

struct alignas(16) WaveLDS {
    float C[NC];
    float gv[NG];    // dN/dx dV
    uint32_t hl[NG]; // dN/dx in two bf16 parts, the high one in the low half
};

// hi/lo split of eight values, converted in pairs (one packed conversion per pair and part)
__device__ inline void split8(const float (&x)[8], bf16x8& hi, bf16x8& lo)
{
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const floatx2 v = {x[2 * p], x[2 * p + 1]};
        const bf16x2 h = __builtin_convertvector(v, bf16x2);
        const floatx2 r = v - __builtin_convertvector(h, floatx2);
        const bf16x2 l = __builtin_convertvector(r, bf16x2);
        hi[2 * p] = h[0];
        hi[2 * p + 1] = h[1];
        lo[2 * p] = l[0];
        lo[2 * p + 1] = l[1];
    }
}

// one element's C on its way to LDS; C is FP64 (the reference's qtensor4) or FP32.  Loads are unconditional
// (lanes past the end re-read the last entry, which store ignores), so that no branch hides them from the
// compiler's wait counting.
template <class TC>
struct StageC;

template <>
struct StageC<double> {
    static constexpr int N = NC / 2, R = (N + 63) / 64; // double2 loads
    double2 v[R];
    __device__ void load(const double* __restrict__ C, int64_t e, int lane)
    {
        const double2* p = reinterpret_cast<const double2*>(C + e * NC);
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = p[min(lane + 64 * k, N - 1)];
    }
    __device__ void store(float* dst, int lane) const
    {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int t = lane + 64 * k;
            if (t < N) {
                dst[2 * t] = static_cast<float>(v[k].x);
                dst[2 * t + 1] = static_cast<float>(v[k].y);
            }
        }
    }
};

template <>
struct StageC<float> {
    static constexpr int N = NC / 4, R = (N + 63) / 64; // 16-byte loads of 4 floats
    floatx4 v[R];
    __device__ void load(const float* __restrict__ C, int64_t e, int lane)
    {
        const floatx4* p = reinterpret_cast<const floatx4*>(C + e * NC);
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = p[min(lane + 64 * k, N - 1)];
    }
    __device__ void store(float* dst, int lane) const
    {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int t = lane + 64 * k;
            if (t < N) *reinterpret_cast<floatx4*>(dst + 4 * t) = v[k];
        }
    }
};

// The 32 x 32 FP32 tile whose top-left 24 x 24 block is K_e of the element with the staged C, gv and hl.
//
// MFMA: lane l supplies A row (l % 32) and B column (l % 32) at contraction slots 8 (l / 32) + s of each
// 16-wide chunk.  The contraction index kk = (q, j2, i) is laid out so that each half-wave h owns
// quadrature points 4h..4h+3: slot s of chunk ch is t = 8 ch + s, q = 4h + t / 9, (j2, i) = t % 9 (t < 36; the
// last 4 slots are zero).  Every index below is then a compile-time constant plus a per-lane base.  Row
// (m, j) of A and column (n, k) of T share the decomposition 3 m + j = 3 n + k, so both operands use
// dNx(q, m, :):  A = delta(j, j2) dNx(q, m, i),  T = sum_l C_q(i, j2, j, l) dV_q dNx(q, m, l).  Rows and
// columns 24..31 are padding, no part of the block: they repeat node 7.
//
// The vector units issue nearly all of the time here, so A comes split from LDS (once per entry instead of
// once per use): a pair of slots is two entries' halves side by side under the lane's mask of j.
__device__ __forceinline__ floatx16 element_tile(const float* C, const float* gv, const uint32_t* hl, int lane)
{
    const int row = lane % 32, h = lane / 32;
    const int j = row % 3, m = row < 24 ? row / 3 : 7;
    const float* Cb = C + h * 4 * 81 + j * 3;
    const float* gb = gv + (h * 4 * NN + m) * 3;
    const uint32_t* ab = hl + (h * 4 * NN + m) * 3;
    // the slots of a pair that are the lane's: both of group j2 = J, or the last of J with the first of J + 1
    const uint32_t both[3] = {j == 0 ? ~0u : 0u, j == 1 ? ~0u : 0u, j == 2 ? ~0u : 0u};
    const uint32_t over[3] = {j == 0 ? 0xFFFFu : j == 1 ? 0xFFFF0000u : 0u, j == 1 ? 0xFFFFu : j == 2 ? 0xFFFF0000u : 0u,
                              j == 2 ? 0xFFFFu : j == 0 ? 0xFFFF0000u : 0u};
    uint32_t a[12]; // the half-wave's 4 points x 3 components
#pragma unroll
    for (int t = 0; t < 12; ++t) a[t] = ab[(t / 3) * 24 + t % 3];
    floatx16 acc = {};
    float g[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ch = 0; ch < KKP / 16; ++ch) {
        float bv[8];
        uint32_t ah[4], al[4];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int t = ch * 8 + s;
            bv[s] = 0.0f;
            if (t < 36) {
                const int ql = t / 9, r = t % 9, j2 = r / 3, i = r % 3;
                if (r == 0) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) g[c] = gb[ql * 24 + c];
                }
                const float* Cq = Cb + ql * 81 + (i * 3 + j2) * 9;
                bv[s] = fmaf(Cq[0], g[0], fmaf(Cq[1], g[1], Cq[2] * g[2]));
                if (s % 2 == 0) {
                    // slots t and t + 1 (35 is odd, so a pair never crosses the end)
                    const int r1 = (t + 1) % 9;
                    const uint32_t lo = a[ql * 3 + i], hi = a[((t + 1) / 9) * 3 + r1 % 3];
                    const uint32_t mask = j2 == r1 / 3 ? both[j2] : over[j2];
                    ah[s / 2] = __builtin_amdgcn_perm(hi, lo, 0x05040100) & mask;
                    al[s / 2] = __builtin_amdgcn_perm(hi, lo, 0x07060302) & mask;
                }
            }
            else if (s % 2 == 0) ah[s / 2] = al[s / 2] = 0u;
        }
        bf16x8 ahi, alo, bhi, blo;
        __builtin_memcpy(&ahi, ah, sizeof(ahi));
        __builtin_memcpy(&alo, al, sizeof(alo));
        split8(bv, bhi, blo);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi, bhi, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi, blo, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(alo, bhi, acc, 0, 0, 0);
    }
    return acc;
}

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Store K_e: the tile's 24 x 24 block goes through LDS (into the staged C, which is no longer read) and
// leaves as one contiguous stream, 16 bytes a lane (VEC: elemmat 16-byte aligned).
// Accumulator layout: value r of lane l is K[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
template <class TK, bool VEC>
__device__ __forceinline__ void store_tile(float* Ks, const floatx16& acc, TK* __restrict__ Ke, int lane)
{
    const int row = lane % 32, h = lane / 32;
    wave_sync();
    if (row < 24) {
#pragma unroll
        for (int r = 0; r < 12; ++r) Ks[(8 * (r / 4) + 4 * h + (r % 4)) * 24 + row] = acc[r];
    }
    wave_sync();
    if constexpr (VEC) {
        constexpr int VW = 16 / static_cast<int>(sizeof(TK)), NV = 576 / VW;
        typedef TK vec __attribute__((ext_vector_type(VW)));
#pragma unroll
        for (int k = 0; k < (NV + 63) / 64; ++k) {
            const int t = lane + 64 * k;
            if (t < NV) {
                vec v;
#pragma unroll
                for (int c = 0; c < VW; ++c) v[c] = static_cast<TK>(Ks[VW * t + c]);
                __builtin_nontemporal_store(v, reinterpret_cast<vec*>(Ke) + t);
            }
        }
    }
    else {
#pragma unroll
        for (int k = 0; k < 9; ++k) Ke[lane + 64 * k] = static_cast<TK>(Ks[lane + 64 * k]);
    }
}

// One wavefront per element, all of whose loads are issued first; many small waves hide them (a wave that
// goes through several elements with the next one's loads in flight measured slower).  Bound by HBM: 6,496
// bytes per element with FP32 arrays (C 2,592, dN/dx and dV 1,600, K_e 2,304).  276,480 elements: 321-333 us,
// 5.4-5.6 TB/s (331-339 us with A split at each use and scalar stores); 140,000: 160 us (173-179); 6,120: 9.4 us
// (11.7).  Forming the geometry from the coordinates saves 1,408 of the bytes and costs more: 323 us with
// one point per lane for eight elements at a time, 350 for four, 386 spread over the wave of each element;
// vector issue and waves in flight are then what is short.
template <class TC, class TK, bool VEC>
__global__ void __launch_bounds__(64 * WAVES) k_stiffness_bf16x3(int64_t nelem, const TC* __restrict__ C,
                                                                 const double* __restrict__ dNx,
                                                                 const double* __restrict__ vol, TK* __restrict__ elemmat)
{
    __shared__ WaveLDS lds[WAVES];
    const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
    WaveLDS& L = lds[w];
    const int64_t e = static_cast<int64_t>(blockIdx.x) * WAVES + w;
    if (e >= nelem) return; // uniform per wave; the kernel has no workgroup barrier
    StageC<TC> st;
    st.load(C, e, lane);
#pragma unroll
    for (int k = 0; k < NG / 64; ++k) {
        const int t = lane + 64 * k;
        const float f = static_cast<float>(dNx[e * NG + t]), v = static_cast<float>(vol[e * NQ + t / 24]);
        const __bf16 hi = static_cast<__bf16>(f), lo = static_cast<__bf16>(f - static_cast<float>(hi));
        L.gv[t] = f * v;
        L.hl[t] = __builtin_bit_cast(uint16_t, hi) | static_cast<uint32_t>(__builtin_bit_cast(uint16_t, lo)) << 16;
    }
    st.store(L.C, lane);
    wave_sync();
    const floatx16 acc = element_tile(L.C, L.gv, L.hl, lane);
    store_tile<TK, VEC>(L.C, acc, elemmat + e * 576, lane);
}

// FP64 in reference order: acc(j, k) += ((dNx(m,i) C(i,j,k,l)) dNx(n,l)) dV over q, i, l.  8 GRP lanes
// per element, 8 / GRP elements per wave: a lane owns node m and 8 / GRP column nodes, so one product
// dNx(m,i) C(i,j,k,l) and one LDS read of C serve 8 / GRP of its blocks, and the same read serves the
// wave's elements.  The tangent and gradients of a point go to registers one point ahead and from there
// to LDS.  Bound by FP64 issue: the order allows no FMA and no regrouping, so an entry costs three
// operations a term plus its share of the first product (3.25 with GRP 2, 3.5 with GRP 4, 4 with GRP 8).
// At 82,861 elements: 395 us (GRP 2; the vector units issue in 83% of its cycles), 414 (GRP 4), 473
// (GRP 8); 507 us for a whole element staged per wave with every lane forming all four operations.
constexpr int SG = 82;      // offset of a point's gradients behind its 81 tangent entries
constexpr int SP = SG + 24; // LDS pitch of an element (its 16-byte reads hit disjoint banks)

template <int LPE> // lanes per element
struct PointStage {
    static constexpr int R = (81 + 24 + LPE - 1) / LPE;
    double r[R];
    double v;
    // point q of element e for lane l of LPE: 81 tangent entries, then the 24 gradients
    __device__ void load(const double* __restrict__ C, const double* __restrict__ dNx, const double* __restrict__ vol,
                         int64_t e, int q, int l)
    {
        const double* c = C + e * NC + q * 81;
        const double* g = dNx + e * NG + q * 24;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int t = l + LPE * k;
            r[k] = t < 81 ? c[t] : g[min(t - 81, 23)];
        }
        v = vol[e * NQ + q];
    }
    __device__ void store(double* dst, int l) const
    {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int t = l + LPE * k;
            if (t < 105) dst[t + (t >= 81)] = r[k];
        }
    }
};

// STREAM: each element matrix leaves through LDS as one contiguous 16-byte stream (elemmat 16-byte
// aligned) instead of scalar stores.
template <int GRP, bool STREAM>
__global__ void __launch_bounds__(64 * WAVES) k_stiffness_f64(int64_t nelem, const double* __restrict__ C,
                                                               const double* __restrict__ dNx,
                                                               const double* __restrict__ vol,
                                                               double* __restrict__ elemmat)
{
    constexpr int LPE = 8 * GRP, EPW = 64 / LPE, NB = 8 / GRP;
    static_assert(EPW * SP <= 576, "the staged points must fit the element matrix");
    __shared__ __align__(16) double lds[WAVES][576];
    const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int s = lane / LPE, l = lane % LPE, m = l / GRP, n0 = NB * (l % GRP);
    double* sh = lds[w];
    double* se = sh + s * SP;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * WAVES * EPW;
    int64_t e0 = (static_cast<int64_t>(blockIdx.x) * WAVES + w) * EPW;
    if (e0 >= nelem) return; // uniform per wave; the kernel has no workgroup barrier
    PointStage<LPE> st;
    st.load(C, dNx, vol, min(e0 + s, nelem - 1), 0, l);
    for (; e0 < nelem; e0 += stride) {
        const int64_t ec = min(e0 + s, nelem - 1), en = min(e0 + stride + s, nelem - 1);
        double acc[NB][3][3] = {};
#pragma unroll 1
        for (int q = 0; q < NQ; ++q) {
            st.store(se, l);
            const double v = st.v;
            wave_sync();
            st.load(C, dNx, vol, q + 1 < NQ ? ec : en, q + 1 < NQ ? q + 1 : 0, l);
            double gm[3], gn[NB][3];
#pragma unroll
            for (int i = 0; i < 3; ++i) gm[i] = se[SG + 3 * m + i];
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int i = 0; i < 3; ++i) gn[n][i] = se[SG + 3 * (n0 + n) + i];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            const double gc = gm[i] * se[((i * 3 + j) * 3 + k) * 3 + d];
#pragma unroll
                            for (int n = 0; n < NB; ++n) acc[n][j][k] += gc * gn[n][d] * v;
                        }
            wave_sync(); // every lane is done reading the point
        }
        if constexpr (STREAM) {
#pragma unroll 1
            for (int t = 0; t < EPW; ++t) {
                if (e0 + t >= nelem) break; // uniform per wave
                if (s == t) {
#pragma unroll
                    for (int j = 0; j < 3; ++j)
#pragma unroll
                        for (int n = 0; n < NB; ++n)
#pragma unroll
                            for (int k = 0; k < 3; ++k) sh[(m * 3 + j) * 24 + (n0 + n) * 3 + k] = acc[n][j][k];
                }
                wave_sync();
                typedef double d2 __attribute__((ext_vector_type(2)));
                d2* Ke = reinterpret_cast<d2*>(elemmat + (e0 + t) * 576);
#pragma unroll
                for (int r = 0; r < 5; ++r)
                    if (r < 4 || lane < 32)
                        __builtin_nontemporal_store(reinterpret_cast<const d2*>(sh)[lane + 64 * r], Ke + lane + 64 * r);
                wave_sync();
            }
        }
        else if (e0 + s < nelem) {
            double* Ke = elemmat + (e0 + s) * 576;
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int k = 0; k < 3; ++k) Ke[(m * 3 + j) * 24 + (n0 + n) * 3 + k] = acc[n][j][k];
        }
    }
}

// out[e] = Ke[e] ue[e]  (batched element GEMV), one thread per element row; an FP32 Ke is widened
// to FP64 before each product
template <class TE>
__global__ void k_elemmat_dot(int64_t nrows, int K, const TE* __restrict__ Ke, const double* __restrict__ ue,
                              double* __restrict__ out)
{
    int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= nrows) return;
    const int64_t e = t / K;
    const TE* row = Ke + t * K;
    const double* x = ue + e * K;
    double s = 0.0;
    for (int c = 0; c < K; ++c) s += static_cast<double>(row[c]) * x[c];
    out[t] = s;
}

// the same product for K = 8 or 24: each wave streams 64 rows (64 K contiguous entries), issuing
// all of its 16-byte loads before using any, multiplies by the element vector (FP64 products),
// stages the products in LDS and sums each row in column order (the order of k_elemmat_dot, so the
// results are identical).  Ke and ue must be 16-byte aligned.
template <int K, class TE, int RW>
__global__ void __launch_bounds__(256) k_elemmat_dot_rows(int64_t nrows, const TE* __restrict__ Ke,
                                                         const double* __restrict__ ue, double* __restrict__ out)
{
    // RW rows per wave: their RW K contiguous entries are loaded by all 64 lanes, 16 bytes at a
    // time, the products go to LDS, and lane l < RW sums row l in column order
    constexpr int VW = 16 / static_cast<int>(sizeof(TE)); // entries per 16-byte load
    static_assert(K % VW == 0, "whole loads per row");
    static_assert((RW * K) % (VW * 64) == 0, "whole loads per wave");
    typedef TE vec __attribute__((ext_vector_type(VW)));
    constexpr int RP = K + 1; // LDS row pitch
    constexpr int NV = RW * K / (VW * 64);
    __shared__ double sh[4][RW * RP];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * 4 + w) * RW;
    if (r0 >= nrows) return; // uniform per wave
    const int64_t base = r0 * K, total = nrows * K;
    const vec* KV = reinterpret_cast<const vec*>(Ke + base);
    vec kv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int loc = VW * (k * 64 + l);
        kv[k] = base + loc < total ? KV[k * 64 + l] : vec{};
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int loc = VW * (k * 64 + l); // a multiple of VW, so loc .. loc + VW - 1 lie in one row
        const int64_t f = base + loc;
        double p[VW];
#pragma unroll
        for (int v = 0; v < VW; ++v) p[v] = 0.0;
        if (f < total) {
            const int64_t e = f / (K * K);
            const int c = static_cast<int>(f % K);
#pragma unroll
            for (int v = 0; v < VW; ++v) p[v] = static_cast<double>(kv[k][v]) * ue[e * K + c + v];
        }
        double* d = sh[w] + (loc / K) * RP + loc % K;
#pragma unroll
        for (int v = 0; v < VW; ++v) d[v] = p[v];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int64_t t = r0 + l;
    if (l < RW && t < nrows) {
        double acc = 0.0;
#pragma unroll
        for (int c = 0; c < K; ++c) acc += sh[w][l * RP + c];
        out[t] = acc;
    }
}

// Lanes per element of k_stiffness_f64: few lanes share most work, but a mesh has to fill the chip with
// them.  Two groups (four elements a wave) from where they are about one full set of resident waves;
// eight (one element a wave) up to where four groups would leave half of the SIMDs without one.  Times in
// us with GRP 2 / 4 / 8: 512 elements 26.1 / 17.0 / 13.3; 2,548: 27.0 / 25.4 / 23.1; 6,120: 43.5 / 36.6 /
// 40.3; 22,680: 113 / 114 / 130; 82,861: 397 / 414 / 473.
constexpr int64_t F64_GRP2 = 16384, F64_GRP4 = 4096;

unsigned grid_for(int64_t nelem, int per_wave = 1)
{
    int64_t g = (nelem + WAVES * per_wave - 1) / (WAVES * per_wave);
    return static_cast<unsigned>(std::min<int64_t>(g, 256 * 64));
}

} // namespace

namespace gf {

template <class TC, class TK>
void launch_bf16x3(gf_quad q, const TC* C, TK* elemmat, hipStream_t s)
{
    GF_REQUIRE(quad_etype(q) == GF_HEX8 && quad_nip(q) == NQ, "GF_BF16X3 needs Hex8 with 8 points");
    GF_REQUIRE(aligned16(C), "GF_BF16X3 needs a 16-byte aligned qtensor4 array");
    const int64_t ne = quad_nelem(q);
    if (ne == 0) return;
    auto kern = aligned16(elemmat) ? k_stiffness_bf16x3<TC, TK, true> : k_stiffness_bf16x3<TC, TK, false>;
    kern<<<nblocks(ne, WAVES), 64 * WAVES, 0, s>>>(ne, C, quad_dNx(q), quad_vol(q), elemmat);
    check_launch();
}

int stiffness_bf16x3(gf_quad q, const double* C, double* elemmat, hipStream_t s)
{
    return guard([&] {
        GF_REQUIRE(aligned16(elemmat), "GF_BF16X3 needs 16-byte aligned qtensor4 and elemmat arrays");
        launch_bf16x3(q, C, elemmat, s);
    });
}

int stiffness_bf16x3_f32(gf_quad q, const float* C, float* elemmat, hipStream_t s)
{
    return guard([&] { launch_bf16x3(q, C, elemmat, s); });
}

int stiffness_f64_hex8(gf_quad q, const double* C, double* elemmat, hipStream_t s)
{
    return guard([&] {
        GF_REQUIRE(quad_etype(q) == GF_HEX8 && quad_nip(q) == NQ, "Hex8 with 8 points");
        const int64_t ne = quad_nelem(q);
        if (ne == 0) return;
        auto run = [&](auto grp) {
            constexpr int G = decltype(grp)::value;
            auto kern = aligned16(elemmat) ? k_stiffness_f64<G, true> : k_stiffness_f64<G, false>;
            kern<<<grid_for(ne, 8 / G), 64 * WAVES, 0, s>>>(ne, C, quad_dNx(q), quad_vol(q), elemmat);
        };
        if (ne >= F64_GRP2) run(std::integral_constant<int, 2>());
        else if (ne >= F64_GRP4) run(std::integral_constant<int, 4>());
        else run(std::integral_constant<int, 8>());
        check_launch();
    });
}

} // namespace gf

namespace {

template <class TE>
int elemmat_dot(int64_t nelem, int K, const TE* elemmat, const double* elemvec, double* out, void* stream)
{
    return guard([&] {
        GF_REQUIRE(elemmat && elemvec && out && K > 0, "invalid argument");
        const int64_t n = nelem * K;
        if (n == 0) return;
        constexpr int RW = 32;                                          // rows per wave
        const unsigned gw = static_cast<unsigned>((n + 4 * RW - 1) / (4 * RW)); // 4 waves per block
        const bool vec = aligned16(elemmat) && aligned16(elemvec);
        if (K == 24 && vec)
            k_elemmat_dot_rows<24, TE, RW><<<gw, 256, 0, S(stream)>>>(n, elemmat, elemvec, out);
        else if (K == 8 && vec)
            k_elemmat_dot_rows<8, TE, RW><<<gw, 256, 0, S(stream)>>>(n, elemmat, elemvec, out);
        else
            k_elemmat_dot<TE><<<nblocks(n, 256), 256, 0, S(stream)>>>(n, K, elemmat, elemvec, out);
        check_launch();
    });
}

} // namespace

extern "C" int gf_elemmat_dot(int64_t nelem, int K, const double* elemmat, const double* elemvec, double* out,
                              void* stream)
{
    return elemmat_dot(nelem, K, elemmat, elemvec, out, stream);
}

extern "C" int gf_elemmat_dot_f32(int64_t nelem, int K, const float* elemmat, const double* elemvec, double* out,
                                  void* stream)
{
    return elemmat_dot(nelem, K, elemmat, elemvec, out, stream);
}

extern "C" int gf_quad_int_gradN_dot_tensor4_dot_gradNT_dV_f32(gf_quad q, const float* qtensor4, float* elemmat,
                                                               void* stream)
{
    return guard([&] {
        GF_REQUIRE(q && qtensor4 && elemmat, "null argument");
        const int rc = gf::stiffness_bf16x3_f32(q, qtensor4, elemmat, S(stream));
        if (rc != GF_OK) throw Error(rc, gf_last_error());
    });
}
