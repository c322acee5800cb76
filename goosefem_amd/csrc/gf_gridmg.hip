// Conjugate gradients preconditioned by a multigrid V-cycle, for the assembled (partitioned or tied)
// operator of a Regular Quad4 grid.
//
// Why: the Jacobi-preconditioned iteration count of these operators grows with the grid's width and each
// iteration is two or three dependent launches of a few microseconds, far from any bandwidth bound.  The
// V-cycle makes the count independent of the grid, for five to a dozen launches per iteration.  Measured
// per solve (one Newton iteration's system, J2 plasticity with most points yielding, Jacobi -> here):
//   plate 24 x 20, 511 -> 26 iterations, 4.6 -> 1.4 ms;  128 x 112, 2,784 -> 28, 28 -> 2.5 ms;
//   300 x 300, 6,927 -> 28, 140 -> 4.9 ms;  tied cell 96 x 96, 2,336 -> 27, 34.7 -> 2.3 ms.
//
// Operator: the condensed matrix on the grid's nodes (opposite edges identified where they are tied or
// share their DOFs) as a 9-point stencil of 2 x 2 blocks, stored as 36 planes [(s 2 + a) 2 + b][node],
// s = (dy + 1) 3 + dx + 1, so that a wave's loads are contiguous and need no column indices.  Rows and
// columns of prescribed components are zero, and so are all vectors there.
//
// Hierarchy: every second grid line (and the last one of an unwrapped direction) is kept; a direction
// of fewer than 6 elements is not coarsened any more.  P is bilinear in the line index, and the coarse
// operators are the Galerkin products P^T A P, again 9-point stencils.  A component that is prescribed
// at a kept node is prescribed on the coarse grid.
//
// Smoother: NS steps of the Chebyshev iteration for M^-1 A on [1 / (1.1 RATIO), 1], M the diagonal of
// absolute row sums: for a symmetric positive definite A the spectrum of M^-1 A lies in (0, 1], on
// every grid and for ragged coarse lines alike, so no eigenvalue estimate is needed and the cycle is a
// symmetric positive definite preconditioner.  The coarsest grid (at most 36 nodes) is solved with its
// dense inverse.
//
// All sums are in a fixed order: a repeated solve gives the same bits.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>

#include "gf_gridlines.hpp"
#include "gf_gridmg.hpp"
#include "gf_wave.hpp"

using namespace gf;

namespace {

constexpr int MAXLEV = 24;
constexpr int NS = 5;             // smoothing steps before and after the coarse correction
constexpr double RATIO = 30.0;    // the smoother's interval
constexpr int TX = 32, TY = 16, NT = TX * TY;             // threads of a smoothing tile
constexpr int HD = NS + 1, HU = NS;                       // its halo: down, up
constexpr int DX = TX - 2 * HD, DY = TY - 2 * HD;         // the nodes it owns: down
constexpr int UX = TX - 2 * HU, UY = TY - 2 * HU;         // up
constexpr int AX = 32, AY = 8, ANT = AX * AY;             // tile of the fine product
constexpr int CT = 256;           // threads of the coarse kernel: its largest grid
constexpr int CMAX = 36;          // nodes of the coarsest grid
constexpr int DT = 1024;          // threads of its inversion
constexpr int CLEV = 8;           // grids that the coarse kernel walks
constexpr int BS = 256;
constexpr int NFOLD = 256;        // partial sums that are left of more than these:
constexpr int FOLD_R = 2048, FOLD_PQ = 1024; // of r.r and r.z; of p.q (k_mg_fold)

// Chebyshev coefficients of the smoother: d = M^-1 r / theta; then d = c1[i] d + c2[i] M^-1 r
struct Cheb {
    double it = 0.0, c1[NS] = {}, c2[NS] = {};
    Cheb()
    {
        const double hi = 1.0, lo = 1.0 / (1.1 * RATIO), th = 0.5 * (hi + lo), de = 0.5 * (hi - lo), sg = th / de;
        double rho = 1.0 / sg;
        it = 1.0 / th;
        for (int i = 1; i < NS; ++i) {
            const double rn = 1.0 / (2.0 * sg - rho);
            c1[i] = rn * rho;
            c2[i] = 2.0 * rn / de;
            rho = rn;
        }
    }
};

struct Level {
    int nx, ny, mx, my, n; // elements, node lines, nodes
    int perx, pery;        // the last line is the first
    int cx, cy;            // the next coarser grid drops every second line of this direction
    double* st;            // [36][n]
    double2* di;           // 1 / sum |row|, 0 where prescribed
    double2 *b, *x, *y;    // right-hand side, the correction before and after the coarser grids'
};

__host__ __device__ inline bool is_line(int f, int n, int per) { return !(f & 1) || (!per && f == n); }

// weights with which fine lines f - 1, f, f + 1 contribute to the coarse line that lies on f
__device__ inline void restrict_weights(int f, int n, int m, int per, int c, double (&w)[3])
{
    const int a = wrap_line(f - 1, m, per), b = wrap_line(f + 1, m, per);
    w[0] = c && a >= 0 && !is_line(a, n, per) ? 0.5 : 0.0;
    w[1] = 1.0;
    w[2] = c && b >= 0 && !is_line(b, n, per) ? 0.5 : 0.0;
}

// fine line of coarse line k
__device__ inline int line_of(int k, int n, int c) { return !c ? k : (2 * k < n ? 2 * k : n); }

// interpolation weight of fine line f (in range) from coarse line k
__device__ inline double weight(int f, int k, int n, int m, int per, int c)
{
    const int p = line_of(k, n, c);
    if (f == p) return 1.0;
    if (!c || is_line(f, n, per)) return 0.0;
    return f == wrap_line(p - 1, m, per) || f == wrap_line(p + 1, m, per) ? 0.5 : 0.0;
}

__device__ inline void load_stencil(const Level& L, int node, double (&S)[36])
{
#pragma unroll
    for (int k = 0; k < 36; ++k) S[k] = L.st[static_cast<int64_t>(k) * L.n + node];
}

// ---- set-up kernels (once per assembled matrix) ----------------------------------------------------

// the finest stencil: each entry from the CSR value it stands for (-1: none)
__global__ void k_mg_gather(int64_t n36, const int32_t* __restrict__ src, const double* __restrict__ val,
                            double* __restrict__ st)
{
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n36) return;
    const int32_t k = src[t];
    st[t] = k >= 0 ? val[k] : 0.0;
}

// ... plus the further values of entries where tied nodes fall together, in CSR order
__global__ void k_mg_gather_more(int64_t n, const int32_t* __restrict__ at, const int32_t* __restrict__ ptr,
                                 const int32_t* __restrict__ src, const double* __restrict__ val,
                                 double* __restrict__ st)
{
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t >= n) return;
    double s = st[at[t]];
    for (int32_t k = ptr[t]; k < ptr[t + 1]; ++k) s += val[src[k]];
    st[at[t]] = s;
}

// M^-1 (absolute row sums)
__global__ void k_mg_diag(Level L)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= L.n) return;
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) s[a] += fabs(L.st[static_cast<int64_t>((k * 2 + a) * 2 + b) * L.n + t]);
    L.di[t] = make_double2(s[0] != 0.0 ? 1.0 / s[0] : 0.0, s[1] != 0.0 ? 1.0 / s[1] : 0.0);
}

// the coarse operator P^T A P: one thread per coarse node and neighbour
__global__ void __launch_bounds__(BS) k_mg_galerkin(Level L, Level C)
{
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= 9 * C.n) return;
    const int s = t / C.n, I = t - s * C.n;
    const int ky = I / C.mx, kx = I - ky * C.mx;
    double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
    const int jx = wrap_line(kx + s % 3 - 1, C.mx, C.perx), jy = wrap_line(ky + s / 3 - 1, C.my, C.pery);
    if (jx >= 0 && jy >= 0) {
        const int px = line_of(kx, L.nx, L.cx), py = line_of(ky, L.ny, L.cy);
        double rx[3], ry[3];
        restrict_weights(px, L.nx, L.mx, L.perx, L.cx, rx);
        restrict_weights(py, L.ny, L.my, L.pery, L.cy, ry);
        for (int i = 0; i < 9; ++i) {
            const double w = rx[i % 3] * ry[i / 3];
            if (w == 0.0) continue;
            const int fx = wrap_line(px + i % 3 - 1, L.mx, L.perx), fy = wrap_line(py + i / 3 - 1, L.my, L.pery);
            double vx[3], vy[3]; // weights of the fine neighbours of (fx, fy) from (jx, jy)
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                const int gx = wrap_line(fx + o - 1, L.mx, L.perx), gy = wrap_line(fy + o - 1, L.my, L.pery);
                vx[o] = gx < 0 ? 0.0 : weight(gx, jx, L.nx, L.mx, L.perx, L.cx);
                vy[o] = gy < 0 ? 0.0 : weight(gy, jy, L.ny, L.my, L.pery, L.cy);
            }
            // all 36 entries at once: a load that waits for its weight waits 36 times
            double S[36];
            load_stencil(L, fy * L.mx + fx, S);
#pragma unroll
            for (int o = 0; o < 9; ++o) {
                const double v = w * vx[o % 3] * vy[o / 3];
                acc[0][0] = fma(v, S[4 * o], acc[0][0]);
                acc[0][1] = fma(v, S[4 * o + 1], acc[0][1]);
                acc[1][0] = fma(v, S[4 * o + 2], acc[1][0]);
                acc[1][1] = fma(v, S[4 * o + 3], acc[1][1]);
            }
        }
        const double2 mi = L.di[py * L.mx + px],
                      mj = L.di[line_of(jy, L.ny, L.cy) * L.mx + line_of(jx, L.nx, L.cx)];
        if (mi.x == 0.0) acc[0][0] = acc[0][1] = 0.0;
        if (mi.y == 0.0) acc[1][0] = acc[1][1] = 0.0;
        if (mj.x == 0.0) acc[0][0] = acc[1][0] = 0.0;
        if (mj.y == 0.0) acc[0][1] = acc[1][1] = 0.0;
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) C.st[static_cast<int64_t>((s * 2 + a) * 2 + b) * C.n + I] = acc[a][b];
}

// Dense inverse of the coarsest operator (prescribed components: the identity), Gauss-Jordan without
// pivoting (symmetric positive definite) in one workgroup.  *unfit = 1 where a pivot is lost to rounding, that
// is below 1e-12 of its diagonal entry (72 rows of sums leave about 1e-14): the operator of a plate or cell
// that is free to move or turn.  Its "inverse" would add a motion of any size to the solution.
__global__ void __launch_bounds__(DT) k_mg_dense(Level C, double* __restrict__ inv, int32_t* __restrict__ unfit)
{
    constexpr int N = 2 * CMAX;
    __shared__ double A[N][N + 1], diag[N];
    const int m = 2 * C.n;
    for (int t = threadIdx.x; t < m * m; t += DT) A[t / m][t % m] = 0.0;
    __syncthreads();
    for (int t = threadIdx.x; t < 9 * C.n; t += DT) {
        const int s = t / C.n, I = t - s * C.n, ky = I / C.mx, kx = I - ky * C.mx;
        const int jx = wrap_line(kx + s % 3 - 1, C.mx, C.perx), jy = wrap_line(ky + s / 3 - 1, C.my, C.pery);
        if (jx < 0 || jy < 0) continue;
        const int J = jy * C.mx + jx;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) A[2 * I + a][2 * J + b] = C.st[static_cast<int64_t>((s * 2 + a) * 2 + b) * C.n + I];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < m; t += DT) {
        if (A[t][t] == 0.0) A[t][t] = 1.0;
        diag[t] = A[t][t];
    }
    if (threadIdx.x == 0) *unfit = 0;
    __syncthreads();
    for (int k = 0; k < m; ++k) {
        if (!(A[k][k] > 1e-12 * diag[k])) { // the same for every thread
            if (threadIdx.x == 0) *unfit = 1;
            return;
        }
        const double pv = 1.0 / A[k][k];
        double v[(N * N + DT - 1) / DT];
#pragma unroll
        for (int j = 0; j < (N * N + DT - 1) / DT; ++j) {
            const int t = threadIdx.x + j * DT;
            v[j] = 0.0;
            if (t >= m * m) continue;
            const int r = t / m, c = t - (t / m) * m;
            if (r == k) v[j] = c == k ? pv : A[k][c] * pv;
            else v[j] = c == k ? -A[r][k] * pv : fma(-A[r][k] * pv, A[k][c], A[r][c]);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < (N * N + DT - 1) / DT; ++j) {
            const int t = threadIdx.x + j * DT;
            if (t < m * m) A[t / m][t - (t / m) * m] = v[j];
        }
        __syncthreads();
    }
    for (int t = threadIdx.x; t < m * m; t += DT) inv[t] = A[t / m][t % m];
}

// ---- the cycle -------------------------------------------------------------------------------------

// r - A d at one node: d of the nine neighbours in LDS at at[s]
__device__ inline double2 minus_product(const double (&S)[36], const double2* d, const int (&at)[3], const int (&dy)[3],
                                        double2 r)
{
#pragma unroll
    for (int s = 0; s < 9; ++s) {
        const double2 v = d[dy[s / 3] + at[s % 3]];
        r.x = fma(-S[4 * s], v.x, fma(-S[4 * s + 1], v.y, r.x));
        r.y = fma(-S[4 * s + 2], v.x, fma(-S[4 * s + 3], v.y, r.y));
    }
    return r;
}

// P e at fine node (fx, fy) of L from the coarse vector e
__device__ inline double2 prolong(const Level& L, const Level& C, const double2* e, int fx, int fy)
{
    int kx[2], ky[2];
    const bool hx = L.cx && !is_line(fx, L.nx, L.perx), hy = L.cy && !is_line(fy, L.ny, L.pery);
    kx[0] = !L.cx ? fx : (is_line(fx, L.nx, L.perx) && (fx & 1) ? C.mx - 1 : fx >> 1);
    ky[0] = !L.cy ? fy : (is_line(fy, L.ny, L.pery) && (fy & 1) ? C.my - 1 : fy >> 1);
    kx[1] = hx ? (kx[0] + 1 < C.mx ? kx[0] + 1 : 0) : kx[0];
    ky[1] = hy ? (ky[0] + 1 < C.my ? ky[0] + 1 : 0) : ky[0];
    const double2 e00 = e[ky[0] * C.mx + kx[0]], e01 = e[ky[0] * C.mx + kx[1]], e10 = e[ky[1] * C.mx + kx[0]],
                  e11 = e[ky[1] * C.mx + kx[1]];
    return make_double2(0.25 * ((e00.x + e01.x) + (e10.x + e11.x)), 0.25 * ((e00.y + e01.y) + (e10.y + e11.y)));
}

// What the finest grid's kernels also do: the conjugate-gradient update before the smoothing (down)
// and the partial sums.
struct Fine {
    const double2 *rold, *q, *p; // r of the last iteration, A p, p (it > 0)
    double2 *rnew, *xsol;
    const double* pq;            // partials of p.q
    int npq;
    double* part;                // partials: r.r (down), r.z (up)
    const double* scal;          // [0], [1] r.z by iteration parity, [4] tol^2 b.b
    int32_t* state;              // [0] done, [1] iterations
    int it;
};

// One grid on the way down: x = NS smoothing steps for b from zero, then the restricted residual.
// A tile of 32 x 16 threads holds its nodes and a halo of NS + 1, each thread one node with its 36
// stencil entries in registers, the Chebyshev direction in LDS: every step needs one ring less, so the
// whole smoothing is one launch.  It owns 20 x 4 of its 512 nodes (22 x 6 on the way up), so each stencil is
// read 6.4 (3.9) times.  On grids of some ten thousand nodes those reads hit the caches, and a launch with its
// dependent loads (5 to 14 us) is the bound; a 1,000 x 1,000 plate takes 1.29 ms per iteration, where reading
// each stencil once per sweep would take some 0.2, so there they are.
// FINE: b is the residual after the conjugate-gradient update, formed on the halo too (r and q are read
// there), and written with x and the partials of r.r for the tile's own nodes.
//
// (*) Workgroup 0 may raise the flag in this launch while waves of others are still to read it.  A wave that
// reads it early must not leave the reduction's barriers to the rest of its workgroup: every wave goes
// through the reduction, and those that read no flag come to the same decision from the same sum.
template <bool FINE>
__global__ void __launch_bounds__(NT) k_mg_down(Level L, Level C, Cheb ch, Fine F, const int32_t* __restrict__ state)
{
    const int done = state[0];
    __shared__ double2 s_d[NT];
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int ux = tile_raw<TX, HD>(blockIdx.x, lx), uy = tile_raw<TY, HD>(blockIdx.y, ly);
    const int gx = tile_line<TX, HD>(blockIdx.x, lx, L.mx, L.perx), gy = tile_line<TY, HD>(blockIdx.y, ly, L.my, L.pery);
    const bool in = gx >= 0 && gy >= 0;
    const int node = in ? gy * L.mx + gx : 0;
    const bool own = lx >= HD && lx < TX - HD && ly >= HD && ly < TY - HD && ux < L.mx && uy < L.my;
    double S[36];
    load_stencil(L, node, S);
    double2 di = L.di[node], r;
    if constexpr (FINE) {
        r = F.rold[node];
        if (F.it > 0) {
            const double2 q = F.q[node];
            double pq = 0.0;
            for (int i = threadIdx.x; i < F.npq; i += NT) pq += F.pq[i];
            pq = block_sum<NT>(pq);
            if (done) return; // (*)
            const double alpha = F.scal[(F.it - 1) & 1] / pq;
            if (!(pq > 0.0)) { // not positive definite (or not a number): the same in every workgroup
                if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) F.state[0] = 4;
                return;
            }
            r.x = fma(-alpha, q.x, r.x);
            r.y = fma(-alpha, q.y, r.y);
            if (own) {
                const double2 p = F.p[node];
                double2 x = F.xsol[node];
                x.x = fma(alpha, p.x, x.x);
                x.y = fma(alpha, p.y, x.y);
                F.xsol[node] = x;
            }
        }
        else if (done) return;
        if (own) F.rnew[node] = r;
        const double rr = block_sum<NT>(own ? r.x * r.x + r.y * r.y : 0.0);
        if (threadIdx.x == 0) F.part[blockIdx.y * gridDim.x + blockIdx.x] = rr;
    }
    else {
        if (done) return;
        r = L.b[node];
    }
    if (!in) {
        r = make_double2(0.0, 0.0);
        di = r;
#pragma unroll
        for (int k = 0; k < 36; ++k) S[k] = 0.0;
    }
    const int at[3] = {max(lx - 1, 0), lx, min(lx + 1, TX - 1)};
    const int dy[3] = {max(ly - 1, 0) * TX, ly * TX, min(ly + 1, TY - 1) * TX};
    double2 d = make_double2(ch.it * (di.x * r.x), ch.it * (di.y * r.y)), x = d;
#pragma unroll
    for (int i = 1; i <= NS; ++i) {
        s_d[threadIdx.x] = d;
        __syncthreads();
        r = minus_product(S, s_d, at, dy, r);
        __syncthreads();
        if (i < NS) {
            d.x = fma(ch.c1[i], d.x, ch.c2[i] * (di.x * r.x));
            d.y = fma(ch.c1[i], d.y, ch.c2[i] * (di.y * r.y));
            x.x += d.x;
            x.y += d.y;
        }
    }
    if (own) L.x[node] = x;
    s_d[threadIdx.x] = r;
    __syncthreads();
    // b_C = P^T r at the coarse nodes that lie on the tile's own nodes
    if (own && (!L.cx || is_line(gx, L.nx, L.perx)) && (!L.cy || is_line(gy, L.ny, L.pery))) {
        const int kx = !L.cx ? gx : ((gx & 1) ? C.mx - 1 : gx >> 1), ky = !L.cy ? gy : ((gy & 1) ? C.my - 1 : gy >> 1);
        double wx[3], wy[3];
        restrict_weights(gx, L.nx, L.mx, L.perx, L.cx, wx);
        restrict_weights(gy, L.ny, L.my, L.pery, L.cy, wy);
        double2 c = make_double2(0.0, 0.0);
#pragma unroll
        for (int s = 0; s < 9; ++s) {
            const double2 v = s_d[(ly + s / 3 - 1) * TX + lx + s % 3 - 1];
            const double w = wx[s % 3] * wy[s / 3];
            c.x = fma(w, v.x, c.x);
            c.y = fma(w, v.y, c.y);
        }
        C.b[ky * C.mx + kx] = make_double2(di.x != 0.0 ? c.x : 0.0, di.y != 0.0 ? c.y : 0.0);
    }
}

// One grid on the way up: x += P e (prescribed components stay zero), then NS smoothing steps; the
// tiles are as on the way down with one ring less.  xin and xout differ, since a tile reads its
// neighbours' nodes.  FINE: b is r, xout is z, with the partials of r.z.
template <bool FINE>
__global__ void __launch_bounds__(NT) k_mg_up(Level L, Level C, Cheb ch, const double2* __restrict__ b,
                                              const double2* __restrict__ e, double2* __restrict__ xout,
                                              double* __restrict__ part, const int32_t* __restrict__ state)
{
    if (state[0]) return;
    __shared__ double2 s_d[NT];
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int ux = tile_raw<TX, HU>(blockIdx.x, lx), uy = tile_raw<TY, HU>(blockIdx.y, ly);
    const int gx = tile_line<TX, HU>(blockIdx.x, lx, L.mx, L.perx), gy = tile_line<TY, HU>(blockIdx.y, ly, L.my, L.pery);
    const bool in = gx >= 0 && gy >= 0;
    const int node = in ? gy * L.mx + gx : 0;
    const bool own = lx >= HU && lx < TX - HU && ly >= HU && ly < TY - HU && ux < L.mx && uy < L.my;
    double S[36];
    load_stencil(L, node, S);
    double2 di = L.di[node], r = b[node], x = L.x[node];
    const double2 rb = r;
    const double2 pe = prolong(L, C, e, in ? gx : 0, in ? gy : 0);
    if (!in) {
        r = make_double2(0.0, 0.0);
        di = x = r;
#pragma unroll
        for (int k = 0; k < 36; ++k) S[k] = 0.0;
    }
    x.x = di.x != 0.0 ? x.x + pe.x : 0.0;
    x.y = di.y != 0.0 ? x.y + pe.y : 0.0;
    const int at[3] = {max(lx - 1, 0), lx, min(lx + 1, TX - 1)};
    const int dy[3] = {max(ly - 1, 0) * TX, ly * TX, min(ly + 1, TY - 1) * TX};
    double2 d = x;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        s_d[threadIdx.x] = d;
        __syncthreads();
        r = minus_product(S, s_d, at, dy, r);
        __syncthreads();
        if (i == 0) d = make_double2(ch.it * (di.x * r.x), ch.it * (di.y * r.y));
        else {
            d.x = fma(ch.c1[i], d.x, ch.c2[i] * (di.x * r.x));
            d.y = fma(ch.c1[i], d.y, ch.c2[i] * (di.y * r.y));
        }
        x.x += d.x;
        x.y += d.y;
    }
    if (own) xout[node] = x;
    if constexpr (FINE) {
        const double rz = block_sum<NT>(own ? rb.x * x.x + rb.y * x.y : 0.0);
        if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = rz;
    }
}

// All grids of at most CT nodes in one workgroup: the rest of the V-cycle for the right-hand side b of
// the first of them, its correction to x.  One thread per node; vectors in LDS.
struct CoarseArgs {
    int nlev;
    Level L[CLEV];
    const double* inv;
};

__global__ void __launch_bounds__(CT) k_mg_coarse(CoarseArgs A, Cheb ch, const int32_t* __restrict__ state)
{
    if (state[0]) return;
    constexpr int TOT = 2 * CT;
    __shared__ double2 s_b[TOT], s_x[TOT], s_d[CT];
    const int t = threadIdx.x;
    // offsets of the grids in s_b and s_x (their sizes shrink at least by a third from grid to grid
    // until the coarsest, which gridmg_create checks against TOT)
    if (t < A.L[0].n) s_b[t] = A.L[0].b[t];
    __syncthreads();
    int off = 0;
    for (int l = 0; l + 1 < A.nlev; ++l) {
        const Level& L = A.L[l];
        const Level& C = A.L[l + 1];
        const bool in = t < L.n;
        const int node = in ? t : 0, gy = node / L.mx, gx = node - gy * L.mx;
        double S[36];
        load_stencil(L, node, S);
        const double2 di = L.di[node];
        int at[3], dy[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            at[o] = max(wrap_line(gx + o - 1, L.mx, L.perx), 0);
            dy[o] = max(wrap_line(gy + o - 1, L.my, L.pery), 0) * L.mx;
        }
        double2 r = s_b[off + node];
        double2 d = make_double2(ch.it * (di.x * r.x), ch.it * (di.y * r.y)), x = d;
#pragma unroll
        for (int i = 1; i <= NS; ++i) {
            if (in) s_d[t] = d;
            __syncthreads();
            r = minus_product(S, s_d, at, dy, r);
            __syncthreads();
            if (i < NS) {
                d.x = fma(ch.c1[i], d.x, ch.c2[i] * (di.x * r.x));
                d.y = fma(ch.c1[i], d.y, ch.c2[i] * (di.y * r.y));
                x.x += d.x;
                x.y += d.y;
            }
        }
        if (in) {
            s_x[off + t] = x;
            s_d[t] = r;
        }
        __syncthreads();
        if (t < C.n) {
            const int ky = t / C.mx, kx = t - ky * C.mx;
            const int px = line_of(kx, L.nx, L.cx), py = line_of(ky, L.ny, L.cy);
            double wx[3], wy[3];
            restrict_weights(px, L.nx, L.mx, L.perx, L.cx, wx);
            restrict_weights(py, L.ny, L.my, L.pery, L.cy, wy);
            int fx[3], fy[3];
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                fx[o] = max(wrap_line(px + o - 1, L.mx, L.perx), 0);
                fy[o] = max(wrap_line(py + o - 1, L.my, L.pery), 0) * L.mx;
            }
            double2 c = make_double2(0.0, 0.0);
#pragma unroll
            for (int s = 0; s < 9; ++s) {
                const double2 v = s_d[fy[s / 3] + fx[s % 3]];
                const double w = wx[s % 3] * wy[s / 3];
                c.x = fma(w, v.x, c.x);
                c.y = fma(w, v.y, c.y);
            }
            const double2 m = C.di[t];
            s_b[off + L.n + t] = make_double2(m.x != 0.0 ? c.x : 0.0, m.y != 0.0 ? c.y : 0.0);
        }
        off += L.n;
        __syncthreads();
    }
    { // the coarsest grid: four lanes per row of the dense inverse
        const Level& L = A.L[A.nlev - 1];
        const int m = 2 * L.n, j = t % 4;
        const double* bb = reinterpret_cast<const double*>(s_b + off);
        for (int row = t / 4; row < 2 * CMAX; row += CT / 4) { // uniform over a row's lanes
            double s = 0.0;
            if (row < m) {
#pragma unroll 6
                for (int c = j; c < m; c += 4) s = fma(A.inv[row * m + c], bb[c], s);
            }
            s += __shfl_xor(s, 1);
            s += __shfl_xor(s, 2);
            if (row < m && j == 0) reinterpret_cast<double*>(s_x + off)[row] = s;
        }
        __syncthreads();
    }
    for (int l = A.nlev - 2; l >= 0; --l) {
        const Level& L = A.L[l];
        const Level& C = A.L[l + 1];
        const int coff = off;
        off -= L.n;
        const bool in = t < L.n;
        const int node = in ? t : 0, gy = node / L.mx, gx = node - gy * L.mx;
        double S[36];
        load_stencil(L, node, S);
        const double2 di = L.di[node];
        int at[3], dy[3];
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            at[o] = max(wrap_line(gx + o - 1, L.mx, L.perx), 0);
            dy[o] = max(wrap_line(gy + o - 1, L.my, L.pery), 0) * L.mx;
        }
        const double2 pe = prolong(L, C, s_x + coff, gx, gy);
        double2 x = s_x[off + node], r = s_b[off + node];
        x.x = di.x != 0.0 ? x.x + pe.x : 0.0;
        x.y = di.y != 0.0 ? x.y + pe.y : 0.0;
        double2 d = x;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if (in) s_d[t] = d;
            __syncthreads();
            r = minus_product(S, s_d, at, dy, r);
            __syncthreads();
            if (i == 0) d = make_double2(ch.it * (di.x * r.x), ch.it * (di.y * r.y));
            else {
                d.x = fma(ch.c1[i], d.x, ch.c2[i] * (di.x * r.x));
                d.y = fma(ch.c1[i], d.y, ch.c2[i] * (di.y * r.y));
            }
            x.x += d.x;
            x.y += d.y;
        }
        if (in) s_x[off + t] = x;
        __syncthreads();
    }
    if (t < A.L[0].n) A.L[0].x[t] = s_x[t];
}

// p = z + beta p_prev on the tile and its ring, q = A p, partials of p.q; block 0 records r.z and the
// iteration count and raises done at convergence (r.r <= tol^2 b.b) or at a breakdown.  The flag is tested
// behind the reduction, as in k_mg_down (*).
__global__ void __launch_bounds__(ANT) k_mg_apply(Level L, const double2* __restrict__ z,
                                                  const double2* __restrict__ pold, double2* __restrict__ pnew,
                                                  double2* __restrict__ q, const double* __restrict__ rr_part, int nrr,
                                                  const double* __restrict__ rz_part, int nrz,
                                                  double* __restrict__ pq_part, double* __restrict__ scal,
                                                  int32_t* __restrict__ state, int it)
{
    const int done = state[0];
    constexpr int HX = AX + 2, HY = AY + 2;
    __shared__ double2 s_p[HX * HY];
    const int lx = threadIdx.x % AX, ly = threadIdx.x / AX;
    const int gx = blockIdx.x * AX + lx, gy = blockIdx.y * AY + ly;
    const bool own = gx < L.mx && gy < L.my;
    const int node = own ? gy * L.mx + gx : 0;
    double S[36];
    load_stencil(L, node, S);
    double2 hz[2], hp[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int t = min(static_cast<int>(threadIdx.x) + j * ANT, HX * HY - 1);
        const int hx = tile_line_ring<HX, 1>(blockIdx.x, t % HX, L.mx, L.perx),
                  hy = tile_line_ring<HY, 1>(blockIdx.y, t / HX, L.my, L.pery);
        const bool ok = hx >= 0 && hy >= 0;
        const int h = ok ? hy * L.mx + hx : 0;
        hz[j] = z[h];
        hp[j] = it > 0 ? pold[h] : make_double2(0.0, 0.0);
        if (!ok) hz[j] = hp[j] = make_double2(0.0, 0.0);
    }
    double rr = 0.0, rz = 0.0, none = 0.0;
    for (int i = threadIdx.x; i < nrr; i += ANT) rr += rr_part[i];
    for (int i = threadIdx.x; i < nrz; i += ANT) rz += rz_part[i];
    block_sum3<ANT>(rr, rz, none);
    if (done) return;
    const bool first = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
    if (first) state[1] = it;
    if (rr <= scal[4] || !(rz > 0.0) || !isfinite(rz)) {
        if (first) state[0] = rr <= scal[4] ? 1 : 4;
        return;
    }
    const double beta = it > 0 ? rz / scal[(it - 1) & 1] : 0.0;
    if (first) scal[it & 1] = rz;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int t = threadIdx.x + j * ANT;
        if (t < HX * HY) s_p[t] = make_double2(fma(beta, hp[j].x, hz[j].x), fma(beta, hp[j].y, hz[j].y));
    }
    __syncthreads();
    const int at[3] = {lx, lx + 1, lx + 2};
    const int dy[3] = {ly * HX, (ly + 1) * HX, (ly + 2) * HX};
    const double2 m = minus_product(S, s_p, at, dy, make_double2(0.0, 0.0));
    const double2 p = s_p[dy[1] + at[1]];
    double c = 0.0;
    if (own) {
        pnew[node] = p;
        q[node] = make_double2(-m.x, -m.y);
        c = -(p.x * m.x + p.y * m.y);
    }
    c = block_sum<ANT>(c);
    if (threadIdx.x == 0) pq_part[blockIdx.y * gridDim.x + blockIdx.x] = c;
}

// Partial sums a (y = 0) and b (y = 1) to NFOLD each, every one of a contiguous share in a fixed order.
// Each workgroup of the kernels that need a sum adds all its partials, so that no launch is spent on it; their
// number and that of the workgroups both grow with the grid, so large grids fold them first.  us per iteration
// of an n x n plate without and with it: n = 500 (5,208 partials of r.r and r.z, 1,008 of p.q) 414-418 and 414,
// folding p.q too 415-418; 600: 467 and 451, with p.q 440; 700: 561 and 530; 1,000: 1,454 and 1,287; 1,500:
// 3,136 and 2,220; 2,000: 8,372 and 5,035.  300 and below: no difference.
__global__ void __launch_bounds__(BS) k_mg_fold(const double* __restrict__ a, int na, const double* __restrict__ b, int nb,
                                                double* __restrict__ out, const int32_t* __restrict__ state)
{
    if (state[0]) return;
    const double* p = blockIdx.y ? b : a;
    const int n = blockIdx.y ? nb : na, share = (n + NFOLD - 1) / NFOLD, e = min((static_cast<int>(blockIdx.x) + 1) * share, n);
    double v = 0.0;
    for (int i = blockIdx.x * share + threadIdx.x; i < e; i += BS) v += p[i];
    v = block_sum<BS>(v);
    if (threadIdx.x == 0) out[blockIdx.y * NFOLD + blockIdx.x] = v;
}

// right-hand side and start on the grid; partials of b.b
__global__ void __launch_bounds__(BS) k_mg_begin(int n, const int32_t* __restrict__ uidx, const double* __restrict__ b,
                                                 const double* __restrict__ x0, double2* __restrict__ rhs,
                                                 double2* __restrict__ x, double* __restrict__ bb_part)
{
    const int t = blockIdx.x * BS + threadIdx.x;
    double bb = 0.0;
    if (t < n) {
        const int32_t u0 = uidx[2 * t], u1 = uidx[2 * t + 1];
        const double2 v = make_double2(u0 >= 0 ? b[u0] : 0.0, u1 >= 0 ? b[u1] : 0.0);
        rhs[t] = v;
        x[t] = x0 ? make_double2(u0 >= 0 ? x0[u0] : 0.0, u1 >= 0 ? x0[u1] : 0.0) : make_double2(0.0, 0.0);
        bb = v.x * v.x + v.y * v.y;
    }
    bb = block_sum<BS>(bb);
    if (threadIdx.x == 0) bb_part[blockIdx.x] = bb;
}

// r = b - A x of a start x
__global__ void __launch_bounds__(BS) k_mg_residual(Level L, const double2* __restrict__ rhs,
                                                    const double2* __restrict__ x, double2* __restrict__ r)
{
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= L.n) return;
    const int gy = t / L.mx, gx = t - gy * L.mx;
    double2 v = rhs[t];
    for (int s = 0; s < 9; ++s) {
        const int jx = wrap_line(gx + s % 3 - 1, L.mx, L.perx), jy = wrap_line(gy + s / 3 - 1, L.my, L.pery);
        if (jx < 0 || jy < 0) continue;
        const double2 p = x[jy * L.mx + jx];
        const double* S = L.st + static_cast<int64_t>(4 * s) * L.n + t;
        v.x = fma(-S[0], p.x, fma(-S[L.n], p.y, v.x));
        v.y = fma(-S[2 * static_cast<int64_t>(L.n)], p.x, fma(-S[3 * static_cast<int64_t>(L.n)], p.y, v.y));
    }
    r[t] = v;
}

__global__ void __launch_bounds__(BS) k_mg_scalars(const double* __restrict__ bb_part, int nbb, double tol,
                                                   double* __restrict__ scal, int32_t* __restrict__ state)
{
    double bb = 0.0;
    for (int i = threadIdx.x; i < nbb; i += BS) bb += bb_part[i];
    bb = block_sum<BS>(bb);
    if (threadIdx.x != 0) return;
    scal[4] = tol * tol * (bb > 0.0 ? bb : 1.0);
    state[0] = !isfinite(bb) ? 2 : state[2] ? 4 : 0; // state[2]: k_mg_dense
    state[1] = 0;
}

__global__ void __launch_bounds__(BS) k_mg_end(int n, const int32_t* __restrict__ uidx, const double2* __restrict__ xg,
                                               double* __restrict__ x)
{
    const int t = blockIdx.x * BS + threadIdx.x;
    if (t >= n) return;
    const double2 v = xg[t];
    const int32_t u0 = uidx[2 * t], u1 = uidx[2 * t + 1];
    if (u0 >= 0) x[u0] = v.x;
    if (u1 >= 0) x[u1] = v.y;
}

} // namespace

namespace gf {

struct GridMG {
    int nlev = 0, first_coarse = 0; // grids, the first one in the coarse kernel
    Level L[MAXLEV];
    int64_t nnu = 0;
    bool stale = true;
    DBuf<double> mem;               // stencils, diagonals and vectors of all grids
    DBuf<int32_t> uidx, src, more_at, more_ptr, more_src, state;
    DBuf<double> part, scal, inv;
    double2 *rhs = nullptr, *xsol = nullptr, *r[2] = {}, *p[2] = {}, *q = nullptr;
    std::unique_ptr<StatePipe> pipe;
    dim3 gdown[MAXLEV], gup[MAXLEV], gapp;
    int nrr = 0, nrz = 0, npq = 0, nbb = 0;
};

void GridMGDelete::operator()(GridMG* m) const { delete m; }

bool gridmg_mesh(const gf_vector_s* v)
{
    if (v->nne != 4 || v->ndim != 2 || v->nelem < 1) return false;
    // conn of Mesh::Quad4::Regular (rows of nx elements, nodes left to right, bottom to top)
    const int64_t N1 = v->conn_h[3], nx = N1 - 1;
    if (nx < 1 || v->nelem % nx != 0) return false;
    const int64_t ny = v->nelem / nx, n = N1 * (ny + 1);
    // 36 n in 32 bits (the stencil's entries); a column of tiles as the y dimension of a launch
    if (n < GRIDMG_MIN_NODES || 36 * n >= INT32_MAX || ny + 1 > 65535 * static_cast<int64_t>(DY) || v->nnode < n) return false;
    for (int64_t e = 0; e < v->nelem; ++e) {
        const int64_t a = (e / nx) * N1 + e % nx, want[4] = {a, a + 1, a + N1 + 1, a + N1};
        for (int m = 0; m < 4; ++m)
            if (v->conn_h[4 * e + m] != want[m]) return false;
    }
    return true;
}

static GridMGPtr build(const gf_vector_s* v, int64_t nnu, const std::function<int64_t(int64_t, int)>& u_of,
                       const std::function<GridMGMatrix()>& matrix, const std::vector<int64_t>& u_of_row)
{
    if (nnu < 1 || !gridmg_mesh(v)) return nullptr;
    const int64_t N1 = v->conn_h[3], nx = N1 - 1, ny = v->nelem / nx;
    // opposite edges stand for the same unknowns: the direction is wrapped
    auto same = [&](int64_t count, int64_t a0, int64_t b0, int64_t step) {
        bool any = false;
        for (int64_t k = 0; k < count; ++k)
            for (int c = 0; c < 2; ++c) {
                const int64_t a = u_of(a0 + k * step, c), b = u_of(b0 + k * step, c);
                if (a != b) return false;
                any |= a >= 0;
            }
        return any;
    };
    const int perx = same(ny + 1, 0, nx, N1), pery = same(N1, 0, ny * N1, 1);
    if ((perx && nx < 6) || (pery && ny < 6)) return nullptr;
    const int mx = static_cast<int>(perx ? nx : N1), my = static_cast<int>(pery ? ny : ny + 1);
    // every unknown belongs to one node and component of the (wrapped) grid
    std::vector<int64_t> at(nnu, -1);
    std::vector<int32_t> uidx(2 * static_cast<size_t>(mx) * my, -2);
    for (int64_t j = 0; j <= ny; ++j)
        for (int64_t i = 0; i <= nx; ++i)
            for (int c = 0; c < 2; ++c) {
                const int64_t u = u_of(j * N1 + i, c);
                const int64_t t = 2 * ((j % my) * mx + i % mx) + c;
                if (u < -1 || u >= nnu) return nullptr;
                if (uidx[t] != -2 && uidx[t] != u) return nullptr;
                uidx[t] = static_cast<int32_t>(u);
                if (u < 0) continue;
                if (at[u] != -1 && at[u] != t) return nullptr;
                at[u] = t;
            }
    for (int64_t u = 0; u < nnu; ++u)
        if (at[u] < 0) return nullptr;
    auto M = GridMGPtr(new GridMG());
    M->nnu = nnu;
    const GridMGMatrix K = matrix();
    const auto &rp = K.rowptr, &cl = K.col;
    // the CSR entry (or entries) behind every stencil entry; rows that stand for different unknowns
    // write different entries, so only rows that share one are kept off the threads
    const int64_t n0 = static_cast<int64_t>(mx) * my;
    struct Place {
        int32_t x, y, t; // grid line numbers, 2 node + component
    };
    std::vector<Place> place(nnu);
    parallel_for(nnu, [&](int64_t u) {
        const int32_t t = static_cast<int32_t>(at[u]), nd = t >> 1, y = nd / mx;
        place[u] = {nd - y * mx, y, t};
    });
    std::vector<int32_t> src(36 * n0, -1);
    std::vector<std::pair<int32_t, int32_t>> more;
    std::mutex guard_more;
    std::atomic<bool> fits{true};
    auto near = [](int d, int m, int per) { // neighbour offset, or 2
        if (per && d > 1) d -= m;
        if (per && d < -1) d += m;
        return d >= -1 && d <= 1 ? d : 2;
    };
    std::vector<char> taken(nnu, 0); // the first row of an unknown fills src, the others go to more
    std::vector<char> first(u_of_row.size(), 0);
    for (size_t r = 0; r < u_of_row.size(); ++r)
        if (u_of_row[r] >= 0 && !taken[u_of_row[r]]) taken[u_of_row[r]] = first[r] = 1;
    parallel_for(static_cast<int64_t>(rp.size()) - 1, [&](int64_t r) {
        const int64_t ur = u_of_row[r];
        if (ur < 0) return;
        const Place pr = place[ur];
        for (int32_t k = rp[r]; k < rp[r + 1]; ++k) {
            const int64_t uc = u_of_row[cl[k]];
            if (uc < 0) continue;
            const Place pc = place[uc];
            const int dx = near(pc.x - pr.x, mx, perx), dy = near(pc.y - pr.y, my, pery);
            if (dx == 2 || dy == 2) {
                fits = false;
                return;
            }
            const int64_t e = ((((dy + 1) * 3 + dx + 1) * 2 + (pr.t & 1)) * 2 + (pc.t & 1)) * n0 + (pr.t >> 1);
            if (first[r] && src[e] < 0) src[e] = k;
            else {
                std::lock_guard<std::mutex> lock(guard_more);
                more.emplace_back(static_cast<int32_t>(e), k);
            }
        }
    });
    if (!fits) return nullptr;
    std::sort(more.begin(), more.end());
    std::vector<int32_t> mat, mptr, msrc;
    for (auto& m : more) {
        if (mat.empty() || mat.back() != m.first) {
            mat.push_back(m.first);
            mptr.push_back(static_cast<int32_t>(msrc.size()));
        }
        msrc.push_back(m.second);
    }
    mptr.push_back(static_cast<int32_t>(msrc.size()));
    // the grids
    std::vector<size_t> off;
    size_t total = 0;
    for (int64_t a = nx, b = ny;;) {
        if (M->nlev == MAXLEV) return nullptr;
        Level& L = M->L[M->nlev++];
        L = Level();
        L.nx = static_cast<int>(a);
        L.ny = static_cast<int>(b);
        L.perx = perx;
        L.pery = pery;
        L.mx = L.nx + (perx ? 0 : 1);
        L.my = L.ny + (pery ? 0 : 1);
        L.n = L.mx * L.my;
        L.cx = a >= 6;
        L.cy = b >= 6;
        off.push_back(total);
        total += (36 + 4 * 2) * static_cast<size_t>(L.n);
        if (!L.cx && !L.cy) break;
        if (L.cx) a = (a + 1) / 2;
        if (L.cy) b = (b + 1) / 2;
    }
    if (M->nlev < 2) return nullptr;
    M->first_coarse = M->nlev - 1;
    size_t held = M->L[M->nlev - 1].n;
    while (M->first_coarse > 1 && M->L[M->first_coarse - 1].n <= CT && M->nlev - M->first_coarse < CLEV &&
           held + M->L[M->first_coarse - 1].n <= 2 * CT)
        held += M->L[--M->first_coarse].n;
    if (M->L[M->nlev - 1].n > CMAX || M->L[M->first_coarse].n > CT) return nullptr;
    const size_t vec0 = total;
    total += 7 * 2 * static_cast<size_t>(n0);
    M->mem.alloc(total);
    for (int l = 0; l < M->nlev; ++l) {
        Level& L = M->L[l];
        L.st = M->mem.p + off[l];
        L.di = reinterpret_cast<double2*>(L.st + 36 * static_cast<size_t>(L.n));
        L.b = L.di + L.n;
        L.x = L.b + L.n;
        L.y = L.x + L.n;
        M->gdown[l] = dim3(nblocks(L.mx, DX), nblocks(L.my, DY));
        M->gup[l] = dim3(nblocks(L.mx, UX), nblocks(L.my, UY));
    }
    double2* w = reinterpret_cast<double2*>(M->mem.p + vec0);
    double2** vecs[] = {&M->rhs, &M->xsol, &M->r[0], &M->r[1], &M->p[0], &M->p[1], &M->q};
    for (auto* p : vecs) {
        *p = w;
        w += n0;
    }
    M->gapp = dim3(nblocks(mx, AX), nblocks(my, AY));
    M->nrr = M->gdown[0].x * M->gdown[0].y;
    M->nrz = M->gup[0].x * M->gup[0].y;
    M->npq = M->gapp.x * M->gapp.y;
    M->nbb = nblocks(n0, BS);
    M->part.alloc(M->nrr + M->nrz + M->npq + M->nbb + 3 * NFOLD);
    M->scal.alloc(8);
    M->state.alloc(4);
    M->inv.alloc(4 * CMAX * CMAX);
    M->uidx.upload(uidx);
    M->src.upload(src);
    M->more_at.upload(mat);
    M->more_ptr.upload(mptr);
    M->more_src.upload(msrc);
    M->pipe = std::make_unique<StatePipe>();
    return M;
}

GridMGPtr gridmg_create(const gf_vector_s* v, int64_t nnu, const std::function<int64_t(int64_t, int)>& u_of,
                        const std::function<GridMGMatrix()>& matrix, const std::vector<int64_t>& u_of_row)
{
    try {
        return build(v, nnu, u_of, matrix, u_of_row);
    }
    catch (const Error& e) {
        if (e.code != GF_ENOMEM) throw;
        (void)hipGetLastError(); // the failed allocation's, which the next launch check would find
    }
    catch (const std::bad_alloc&) {
    }
    return nullptr;
}

void gridmg_invalidate(GridMG* m)
{
    if (m) m->stale = true;
}

static void refresh(GridMG* M, const double* val, hipStream_t s)
{
    const int64_t n36 = 36 * static_cast<int64_t>(M->L[0].n);
    k_mg_gather<<<nblocks(n36, BS), BS, 0, s>>>(n36, M->src.p, val, M->L[0].st);
    if (M->more_at.n)
        k_mg_gather_more<<<nblocks(M->more_at.n, BS), BS, 0, s>>>(M->more_at.n, M->more_at.p, M->more_ptr.p,
                                                                  M->more_src.p, val, M->L[0].st);
    for (int l = 0; l < M->nlev; ++l) {
        if (l) k_mg_galerkin<<<nblocks(9 * static_cast<int64_t>(M->L[l].n), BS), BS, 0, s>>>(M->L[l - 1], M->L[l]);
        k_mg_diag<<<nblocks(M->L[l].n, BS), BS, 0, s>>>(M->L[l]);
    }
    k_mg_dense<<<1, DT, 0, s>>>(M->L[M->nlev - 1], M->inv.p, M->state.p + 2);
    check_launch();
    M->stale = false;
}

GridMGStatus gridmg_solve(GridMG* M, const double* val, const double* b, double* x, bool warm, double tol,
                          int64_t maxiter, int64_t* iterations, hipStream_t s)
{
    const int n0 = M->L[0].n, fc = M->first_coarse;
    if (M->stale) refresh(M, val, s);
    double *rr = M->part.p, *rz = rr + M->nrr, *pq = rz + M->nrz, *bb = pq + M->npq, *fold = bb + M->nbb;
    const bool fold_r = M->nrr + M->nrz > FOLD_R, fold_pq = M->npq > FOLD_PQ;
    int32_t* state = M->state.p;
    static const Cheb ch;
    CoarseArgs ca;
    ca.nlev = M->nlev - fc;
    for (int l = 0; l < ca.nlev; ++l) ca.L[l] = M->L[fc + l];
    ca.inv = M->inv.p;
    k_mg_begin<<<M->nbb, BS, 0, s>>>(n0, M->uidx.p, b, warm ? x : nullptr, M->rhs, M->xsol, bb);
    k_mg_scalars<<<1, BS, 0, s>>>(bb, M->nbb, tol, M->scal.p, state);
    if (warm) k_mg_residual<<<M->nbb, BS, 0, s>>>(M->L[0], M->rhs, M->xsol, M->r[1]);
    // The cycle smooths ten times with a scaled diagonal, so an iteration does the work of at least some seven of the
    // Jacobi iteration and takes the time of about seven, however badly the matrix is scaled: there is no count from
    // which the caller's iteration would be the better one.  128 x 112 plate, iterations and ms, here / Jacobi:
    // one phase 10, 1.0 / 1,389, 13.7; K/G = 10^4 261, 18 / 30,572, 297; log-normal moduli over four decades (one
    // sigma two) to 1e-7 2,111, 146 / 127,284, 1,257; stripes of contrast 10^6 across the load 1,034, 72 /
    // 9,093, 90; elements 100 times as wide as high 165, 12 / 1,331, 13.  The least favourable: such stripes on
    // 64 x 64, 223, 14.0 / 1,408, 13.1.  The cap is for matrices that rounding keeps from converging, on which
    // the caller's iteration mostly fails too: an eighth of its own count.
    // The flag is looked at every 4 iterations, one look behind.
    const int cap = static_cast<int>(std::min<int64_t>(maxiter, std::max<int64_t>(1000, maxiter / 8)));
    constexpr int check_every = 4;
    int32_t st[2] = {0, 0};
    StatePipe& pipe = *M->pipe;
    int chunk = 0;
    for (int it = 0; it <= cap && !st[0];) {
        for (int k = 0; k < check_every && it <= cap; ++k, ++it) {
            Fine F = {};
            F.rold = it > 0 || warm ? M->r[(it + 1) & 1] : M->rhs;
            F.q = M->q;
            F.p = M->p[(it + 1) & 1];
            F.rnew = M->r[it & 1];
            F.xsol = M->xsol;
            F.pq = fold_pq ? fold + 2 * NFOLD : pq;
            F.npq = fold_pq ? NFOLD : M->npq;
            F.part = rr;
            F.scal = M->scal.p;
            F.state = state;
            F.it = it;
            k_mg_down<true><<<M->gdown[0], NT, 0, s>>>(M->L[0], M->L[1], ch, F, state);
            for (int l = 1; l < fc; ++l)
                k_mg_down<false><<<M->gdown[l], NT, 0, s>>>(M->L[l], M->L[l + 1], ch, Fine(), state);
            k_mg_coarse<<<1, CT, 0, s>>>(ca, ch, state);
            const double2* e = M->L[fc].x;
            for (int l = fc - 1; l > 0; --l) {
                k_mg_up<false><<<M->gup[l], NT, 0, s>>>(M->L[l], M->L[l + 1], ch, M->L[l].b, e, M->L[l].y, nullptr, state);
                e = M->L[l].y;
            }
            k_mg_up<true><<<M->gup[0], NT, 0, s>>>(M->L[0], M->L[1], ch, M->r[it & 1], e, M->L[0].y, rz, state);
            if (fold_r) k_mg_fold<<<dim3(NFOLD, 2), BS, 0, s>>>(rr, M->nrr, rz, M->nrz, fold, state);
            k_mg_apply<<<M->gapp, ANT, 0, s>>>(M->L[0], M->L[0].y, M->p[(it + 1) & 1], M->p[it & 1], M->q,
                                               fold_r ? fold : rr, fold_r ? NFOLD : M->nrr, fold_r ? fold + NFOLD : rz,
                                               fold_r ? NFOLD : M->nrz, pq, M->scal.p, state, it);
            if (fold_pq) k_mg_fold<<<NFOLD, BS, 0, s>>>(pq, M->npq, nullptr, 0, fold + 2 * NFOLD, state);
        }
        check_launch();
        pipe.post(state, chunk, s);
        if (chunk > 0) st[0] = pipe.wait(chunk - 1)[0];
        ++chunk;
    }
    const int32_t* last = pipe.wait(chunk - 1);
    st[0] = last[0];
    st[1] = last[1];
    if (iterations) *iterations = st[1];
    if (st[0] == 2) return GRIDMG_BAD_RHS;
    if (st[0] == 4 && st[1] == 0 && warm) // a start that is not finite: solve from zero instead
        return gridmg_solve(M, val, b, x, false, tol, maxiter, iterations, s);
    if (st[0] != 1) return GRIDMG_GAVE_UP;
    k_mg_end<<<M->nbb, BS, 0, s>>>(n0, M->uidx.p, M->xsol, x);
    check_launch();
    return GRIDMG_CONVERGED;
}

} // namespace gf
