// Multigrid-preconditioned conjugate gradients on the assembled operator of a Regular Quad4 grid
// (gf_gridmg.hip): the solve path of the partitioned and the tied sparse matrices on such grids.
#pragma once

#include <functional>
#include <memory>
#include <vector>

#include "gf_internal.hpp"

namespace gf {

struct GridMG;
struct GridMGDelete {
    void operator()(GridMG* m) const;
};
using GridMGPtr = std::unique_ptr<GridMG, GridMGDelete>;

// The mesh is a Regular Quad4 grid of a size that the method takes: at least GRIDMG_MIN_NODES nodes.
// 64: a plate of 11 x 9 nodes takes 0.87 ms per solve instead of 1.8 ms (20 iterations of 30 us against
// 180 of 10 us); a few ten nodes take a few ten of the cheap Jacobi iterations.
constexpr int64_t GRIDMG_MIN_NODES = 64;
bool gridmg_mesh(const gf_vector_s* v);

// The matrix's CSR on the host, asked for once the mesh and the numbering fit.
struct GridMGMatrix {
    std::vector<int32_t> rowptr, col;
};

// Set-up (host), by the first solve: a matrix that is only assembled and multiplied carries none of it (some
// 700 bytes per node).  u_of(node, c): the unknown that component c of a mesh node stands for (shared by
// tied nodes), or -1 if it is prescribed.  The operator's entries are those of the CSR whose row and column r
// stand for the unknown u_of_row[r] (-1: dropped); entries that fall together add up.
// Returns null where the method does not apply (not gridmg_mesh, unknowns that are not one per grid node and
// component after identifying opposite edges, an entry that couples nodes that are not neighbours), and
// where the memory for it is not to be had: the caller's iteration needs none of it.
GridMGPtr gridmg_create(const gf_vector_s* v, int64_t nnu, const std::function<int64_t(int64_t, int)>& u_of,
                        const std::function<GridMGMatrix()>& matrix, const std::vector<int64_t>& u_of_row);

// The matrix values changed (the hierarchy is rebuilt by the next solve).
void gridmg_invalidate(GridMG* m);

enum GridMGStatus { GRIDMG_CONVERGED = 0, GRIDMG_BAD_RHS = 1, GRIDMG_GAVE_UP = 2 };

// x (in: the start, if warm; out: the solution) of A x = b to a recursive residual of tol ||b||, val the
// values of the CSR.  GRIDMG_GAVE_UP: a breakdown (the operator or a start is not fit for the method) or
// the cap on the iterations; x is then as it was.  Waits for the stream up to the last iteration; the copy
// to x is queued behind it.
GridMGStatus gridmg_solve(GridMG* m, const double* val, const double* b, double* x, bool warm, double tol,
                          int64_t maxiter, int64_t* iterations, hipStream_t s);

} // namespace gf
