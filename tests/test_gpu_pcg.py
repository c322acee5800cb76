"""Tied-system PCG on the GPU: the matrix-free K' and K'_up of MatrixPartitionedTyings against a
dense restatement built from the oracle's element stiffness, the reordered [u, p, d] dofs and the
tying matrices; the solve against a direct dense solve, with the true residual as the criterion."""

import numpy as np
import pytest

import oracle
from oracle import HEX8, QUAD4_PLANAR

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gf():
    import goosefem_amd

    goosefem_amd.lib()
    return goosefem_amd


def host(t):
    import torch

    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def periodic_system(gf, et, n, seed=1, square=False):
    if et == HEX8:
        mesh = gf.Mesh.Hex8.Regular(n, n, n)
    else:
        mesh = gf.Mesh.Quad4.Regular(n if square else n + 2, n)
    coor, conn = mesh.coor, mesh.conn
    ctrl = gf.Tyings.Control(coor, mesh.dofs)
    iip = np.concatenate((ctrl.controlDofs.ravel(), ctrl.dofs[mesh.nodesOrigin]))
    ty = gf.Tyings.Periodic(ctrl.coor, ctrl.dofs, ctrl.controlDofs, mesh.nodesPeriodic, iip)
    vec = gf.Vector(conn, ty.dofs)
    nd = coor.shape[1]
    ov = oracle.Vector(conn, oracle.dofs(coor.shape[0], nd))
    x = ov.AsElement(coor)
    oq = oracle.Quadrature(et, x)
    quad = (gf.Element.Hex8.Quadrature(x) if et == HEX8 else gf.Element.Quad4.QuadraturePlanar(x))
    rng = np.random.default_rng(seed)
    G = np.exp(0.4 * rng.standard_normal(oq.nelem))
    K = np.full(oq.nelem, 10.0)
    P = gf.TyingsPCG(vec, quad, K, G, ty)
    # dense reference: A in the [u, p, d] numbering, then the reference's condensation
    C = oracle.elastic_tangent(np.repeat(K[:, None], oq.nip, 1), np.repeat(G[:, None], oq.nip, 1))
    Ke = oq.Int_gradN_dot_tensor4_dot_gradNT_dV(C)
    ndof = ty.nni + ty.nnd
    A = np.zeros((ndof, ndof))
    for e in range(oq.nelem):
        d = ty.dofs[conn[e]].ravel()
        A[np.ix_(d, d)] += Ke[e]
    u, p, dd = slice(0, ty.nnu), slice(ty.nnu, ty.nni), slice(ty.nni, ndof)
    Cdu, Cdp = ty.Cdu, ty.Cdp
    Kp = A[u, u] + A[u, dd] @ Cdu + Cdu.T @ A[dd, u] + Cdu.T @ A[dd, dd] @ Cdu
    Kup = A[u, p] + A[u, dd] @ Cdp + Cdu.T @ A[dd, p] + Cdu.T @ A[dd, dd] @ Cdp
    return mesh, ty, P, Kp, Kup


@pytest.mark.parametrize("et,n", [(QUAD4_PLANAR, 6), (HEX8, 3)])
def test_operator_matches_dense_condensation(gf, et, n):
    mesh, ty, P, Kp, Kup = periodic_system(gf, et, n)
    rng = np.random.default_rng(2)
    xu = rng.standard_normal(ty.nnu)
    xp = rng.standard_normal(ty.nnp)
    y = host(P.apply(xu))
    assert np.linalg.norm(y - Kp @ xu) / np.linalg.norm(Kp @ xu) < 1e-13
    y = host(P.apply(None, xp))
    assert np.linalg.norm(y - Kup @ xp) / np.linalg.norm(Kup @ xp) < 1e-13
    assert np.allclose(host(P.inverse_diagonal), 1.0 / np.diag(Kp), rtol=1e-13)
    full = host(P.expand(xu, xp))
    assert np.array_equal(full[: ty.nnu], xu) and np.array_equal(full[ty.nnu:ty.nni], xp)
    assert np.allclose(full[ty.nni:], ty.Cdu @ xu + ty.Cdp @ xp, rtol=1e-14, atol=1e-14)


@pytest.mark.parametrize("et,n", [(QUAD4_PLANAR, 10), (HEX8, 4)])
def test_solve_matches_direct_and_true_residual(gf, et, n):
    mesh, ty, P, Kp, Kup = periodic_system(gf, et, n)
    xp = np.zeros(ty.nnp)
    xp[ty.control[0, 1] - ty.nnu] = 1e-3  # simple shear increment through ctrl(0, 1)
    b = -host(P.apply(None, xp))
    assert np.linalg.norm(b + Kup @ xp) / np.linalg.norm(Kup @ xp) < 1e-13
    x, it, res = P.solve(b, tol=1e-10)
    x = host(x)
    xd = np.linalg.solve(Kp, b)
    assert res <= 1e-10 * 10
    assert np.linalg.norm(b - Kp @ x) / np.linalg.norm(b) < 1e-9
    assert np.linalg.norm(x - xd) / np.linalg.norm(xd) < 1e-7
    assert 0 < it < 10 * ty.nnu
    # warm start from the solution: converged at once
    x2, it2, res2 = P.solve(b, x0=xd, tol=1e-10)
    assert it2 == 0 and res2 < 1e-10
    # deterministic: a second solve gives identical bits
    x3, it3, _ = P.solve(b, tol=1e-10)
    assert it3 == it and np.array_equal(host(x3), x)


def test_iteration_cap_reports_nonconvergence(gf):
    mesh, ty, P, Kp, Kup = periodic_system(gf, QUAD4_PLANAR, 10)
    b = np.random.default_rng(0).standard_normal(ty.nnu)
    with pytest.raises(gf.GooseFEMError) as e:
        P.solve(b, tol=1e-12, maxiter=3)
    assert e.value.code == gf.GF_ENOTCONV
    x, it, res = P.solve(b, tol=1e-12, maxiter=3, raise_on_fail=False)
    assert it == 3 and res > 1e-12


def test_structured_periodic_operator_and_solve(gf):
    """Square Quad4 cell (n = 32): the fused structured operator (torus element assembly from one
    shared geometry) against the dense condensation, and its solve against the direct solution."""
    mesh, ty, P, Kp, Kup = periodic_system(gf, QUAD4_PLANAR, 32, square=True)
    assert P.structured
    rng = np.random.default_rng(5)
    xu = rng.standard_normal(ty.nnu)
    y = host(P.apply(xu))
    assert np.linalg.norm(y - Kp @ xu) / np.linalg.norm(Kp @ xu) < 1e-13
    xp = np.zeros(ty.nnp)
    xp[ty.control[0, 1] - ty.nnu] = 1e-3
    b = -Kup @ xp
    # the K'_up x_p term goes through the general path (x_p non-zero)
    assert np.linalg.norm(host(P.apply(None, xp)) - Kup @ xp) / np.linalg.norm(Kup @ xp) < 1e-13
    x, it, res = P.solve(b, tol=1e-10)
    x = host(x)
    xd = np.linalg.solve(Kp, b)
    assert res <= 1e-9 and np.linalg.norm(b - Kp @ x) / np.linalg.norm(b) < 1e-9
    assert np.linalg.norm(x - xd) / np.linalg.norm(xd) < 1e-6
    x2, it2, _ = P.solve(b, tol=1e-10)
    assert it2 == it and np.array_equal(host(x2), x)
    # the fused two-launch iteration honours the cap and warm starts
    _, it3, res3 = P.solve(b, tol=1e-12, maxiter=3, raise_on_fail=False)
    assert it3 == 3 and res3 > 1e-12
    _, it4, res4 = P.solve(b, x0=xd, tol=1e-10)
    assert it4 == 0 and res4 < 1e-10
    # the non-square cell of the other tests stays on the general path
    _, _, P2, _, _ = periodic_system(gf, QUAD4_PLANAR, 6)
    assert not P2.structured


def test_structured_periodic_hex8_operator_and_solve(gf):
    """Hex8 cube (n = 8): the structured operator (K_e = K KK + G KG from one shared geometry,
    node-centric sums over the 8 elements of each node) against the dense condensation, and its solve
    against the direct solution."""
    mesh, ty, P, Kp, Kup = periodic_system(gf, HEX8, 8)
    assert P.structured
    rng = np.random.default_rng(6)
    xu = rng.standard_normal(ty.nnu)
    y = host(P.apply(xu))
    assert np.linalg.norm(y - Kp @ xu) / np.linalg.norm(Kp @ xu) < 1e-13
    xp = np.zeros(ty.nnp)
    xp[ty.control[0, 1] - ty.nnu] = 5e-4
    xp[ty.control[1, 0] - ty.nnu] = 5e-4
    b = -Kup @ xp
    x, it, res = P.solve(b, tol=1e-10)
    x = host(x)
    xd = np.linalg.solve(Kp, b)
    assert res <= 1e-9 and np.linalg.norm(b - Kp @ x) / np.linalg.norm(b) < 1e-9
    assert np.linalg.norm(x - xd) / np.linalg.norm(xd) < 1e-6
    x2, it2, _ = P.solve(b, tol=1e-10)
    assert it2 == it and np.array_equal(host(x2), x)
    _, it3, res3 = P.solve(b, tol=1e-12, maxiter=3, raise_on_fail=False)
    assert it3 == 3 and res3 > 1e-12
    _, it4, res4 = P.solve(b, x0=xd, tol=1e-10)
    assert it4 == 0 and res4 < 1e-10


@pytest.mark.parametrize("et,n,square", [(QUAD4_PLANAR, 32, True), (QUAD4_PLANAR, 10, False), (HEX8, 8, False)])
def test_bad_start_falls_back(gf, et, n, square):
    """A learned (or any) start whose residual is not finite or larger than ||b|| is replaced by the
    previous converged solution, if that one does better than zero, else by zero: NaN, 1e6-scaled
    and random starts reach the true residual 1e-10 in the plain solve's iteration count (the zero
    fallback repeats the plain solve bit for bit); a non-finite right-hand side fails at once."""
    mesh, ty, P, Kp, Kup = periodic_system(gf, et, n, square=square)
    xp = np.zeros(ty.nnp)
    xp[ty.control[0, 1] - ty.nnu] = 1e-3
    b = -Kup @ xp
    xd = np.linalg.solve(Kp, b)
    rng = np.random.default_rng(11)
    starts = {
        "nan": np.full(ty.nnu, np.nan),
        "scaled": 1e6 * xd,
        "random": np.abs(xd).max() * rng.standard_normal(ty.nnu),
    }
    x_plain = it_plain = None
    for name, x0 in starts.items():
        # a fresh solver has no previous solution: the fallback is zero, i.e. the plain solve
        _, _, Q, _, _ = periodic_system(gf, et, n, square=square)
        if x_plain is None:
            xz, it_plain, _ = Q.solve(b, tol=1e-10)
            x_plain = host(xz)
            assert Q.start_used == gf.GF_START_GIVEN
            _, _, Q, _, _ = periodic_system(gf, et, n, square=square)
        x, it, res = Q.solve(b, x0=x0, tol=1e-10)
        x = host(x)
        assert Q.start_used == gf.GF_START_ZERO, name
        assert res <= 1e-10 and np.linalg.norm(b - Kp @ x) / np.linalg.norm(b) < 1e-9, name
        assert it == it_plain and np.array_equal(x, x_plain), name
    # with a previous solution: a doubled load from a NaN start restarts from that solution, whose
    # residual is half of ||b||, and needs no more iterations than the plain solve
    P.solve(b, tol=1e-10)
    x, it, res = P.solve(2.0 * b, x0=np.full(ty.nnu, np.nan), tol=1e-10)
    assert P.start_used == gf.GF_START_PREVIOUS
    assert res <= 1e-10 and it <= it_plain
    assert np.linalg.norm(host(x) - 2.0 * xd) / np.linalg.norm(2.0 * xd) < 1e-6
    # a good start is kept
    P.solve(b, x0=xd + 1e-6 * np.abs(xd).max() * rng.standard_normal(ty.nnu), tol=1e-10)
    assert P.start_used == gf.GF_START_GIVEN
    # a non-finite right-hand side is rejected before any iteration
    bad = b.copy()
    bad[3] = np.inf
    with pytest.raises(gf.GooseFEMError) as e:
        P.solve(bad, tol=1e-10)
    assert e.value.code == gf.GF_EINVAL


@pytest.mark.parametrize("size", [(8, 8), (9, 33), (33, 9), (31, 8), (32, 15), (65, 17), (4, 4, 4), (5, 9, 6), (9, 8, 5),
                                  (17, 4, 7), (8, 16, 4)])
def test_structured_operator_of_any_size(gf, size):
    """The structured operators on cells that are no multiple of their tiles (32 x 8 and 8 x 8 x 4 nodes):
    the product against the sum of the oracle's element matrices over the wrapped grid (1e-13: FP64 sums
    of some ten terms), and the solve's residual with that matrix."""
    import scipy.sparse as sp

    nd = len(size)
    et = QUAD4_PLANAR if nd == 2 else HEX8
    mesh = gf.Mesh.Quad4.Regular(*size) if nd == 2 else gf.Mesh.Hex8.Regular(*size)
    coor, conn = mesh.coor, mesh.conn
    ctrl = gf.Tyings.Control(coor, mesh.dofs)
    iip = np.concatenate((ctrl.controlDofs.ravel(), ctrl.dofs[mesh.nodesOrigin]))
    ty = gf.Tyings.Periodic(ctrl.coor, ctrl.dofs, ctrl.controlDofs, mesh.nodesPeriodic, iip)
    x = oracle.Vector(conn, oracle.dofs(coor.shape[0], nd)).AsElement(coor)
    oq = oracle.Quadrature(et, x)
    quad = gf.Element.Hex8.Quadrature(x) if nd == 3 else gf.Element.Quad4.QuadraturePlanar(x)
    rng = np.random.default_rng(sum(size))
    G, K = np.exp(0.4 * rng.standard_normal(oq.nelem)), rng.uniform(5.0, 15.0, oq.nelem)
    P = gf.TyingsPCG(gf.Vector(conn, ty.dofs), quad, K, G, ty)
    assert P.structured
    C = oracle.elastic_tangent(np.repeat(K[:, None], oq.nip, 1), np.repeat(G[:, None], oq.nip, 1))
    Ke = oq.Int_gradN_dot_tensor4_dot_gradNT_dV(C)
    # u-DOF of every node's periodic image; prescribed ones (the origin) get the spare number nnu
    i = np.rint(coor).astype(int) % np.array(size)
    image = np.zeros(coor.shape[0], dtype=int)
    grid = {tuple(r): n for n, r in reversed(list(enumerate(np.rint(coor).astype(int))))}
    for n, r in enumerate(i):
        image[n] = grid[tuple(r)]
    u = np.minimum(ty.dofs[image], ty.nnu)
    d = u[conn].reshape(mesh.nelem, -1)
    k = d.shape[1]
    A = sp.csr_matrix((Ke.ravel(), (np.repeat(d, k, axis=1).ravel(), np.tile(d, (1, k)).ravel())),
                      shape=(ty.nnu + 1,) * 2)[: ty.nnu, : ty.nnu]
    xu = rng.standard_normal(ty.nnu)
    y = host(P.apply(xu))
    assert np.linalg.norm(y - A @ xu) <= 1e-13 * np.linalg.norm(A @ xu)
    b = A @ xu
    sol, it, res = P.solve(b, tol=1e-10)
    assert res <= 1e-9 and np.linalg.norm(b - A @ host(sol)) <= 1e-9 * np.linalg.norm(b)
    again, it2, _ = P.solve(b, tol=1e-10)
    assert it2 == it and np.array_equal(host(again), host(sol))


def tied_cell(gf, size, merge=(), spare=0):
    """A Regular periodic cell (origin fixed) in the numbering [u | p | d], as a program may pass it:
    unknowns of each group in merge are made one, and `spare` nodes that no element uses bring two or three
    unknowns each.  (mesh, vector, quadrature, moduli, tyings, dense K' from the element matrices at coor)"""
    from types import SimpleNamespace

    nd = len(size)
    mesh = gf.Mesh.Quad4.Regular(*size) if nd == 2 else gf.Mesh.Hex8.Regular(*size)
    ctrl = gf.Tyings.Control(mesh.coor, mesh.dofs)
    iip = np.concatenate((ctrl.controlDofs.ravel(), ctrl.dofs[mesh.nodesOrigin]))
    ty = gf.Tyings.Periodic(ctrl.coor, ctrl.dofs, ctrl.controlDofs, mesh.nodesPeriodic, iip)
    drop = np.sort([m for group in merge for m in group[1:]]).astype(np.int64)
    new = np.arange(ty.nni + ty.nnd)
    for group in merge:
        new[list(group[1:])] = group[0]
    new = new - np.searchsorted(drop, new)
    nnu = ty.nnu - drop.size
    new[ty.nnu:] += nd * spare
    dofs = np.concatenate((new[ty.dofs], (nnu + np.arange(nd * spare)).reshape(spare, nd)))
    rp, col, val = ty.Cdu_csr[:3]
    tyings = SimpleNamespace(nnu=nnu + nd * spare, nnp=ty.nnp, nnd=ty.nnd, Cdu_csr=(rp, new[col], val),
                             Cdp_csr=ty.Cdp_csr)
    vec = gf.Vector(mesh.conn, dofs)
    x = oracle.Vector(mesh.conn, oracle.dofs(mesh.nnode, nd)).AsElement(mesh.coor)
    quad = gf.Element.Hex8.Quadrature(x) if nd == 3 else gf.Element.Quad4.QuadraturePlanar(x)
    rng = np.random.default_rng(sum(size))
    K, G = rng.uniform(5.0, 15.0, mesh.nelem), np.exp(0.4 * rng.standard_normal(mesh.nelem))

    def dense(coor):
        et = HEX8 if nd == 3 else QUAD4_PLANAR
        oq = oracle.Quadrature(et, oracle.Vector(mesh.conn, oracle.dofs(mesh.nnode, nd)).AsElement(coor))
        C = oracle.elastic_tangent(np.repeat(K[:, None], oq.nip, 1), np.repeat(G[:, None], oq.nip, 1))
        Ke = oq.Int_gradN_dot_tensor4_dot_gradNT_dV(C)
        nni = tyings.nnu + tyings.nnp
        A = np.zeros((nni + tyings.nnd,) * 2)
        for e in range(mesh.nelem):
            d = dofs[mesh.conn[e]].ravel()
            np.add.at(A, np.ix_(d, d), Ke[e])
        T = np.zeros((tyings.nnd, tyings.nnu))
        for r in range(tyings.nnd):
            T[r, new[col[rp[r]:rp[r + 1]]]] += val[rp[r]:rp[r + 1]]
        u, d = slice(0, tyings.nnu), slice(nni, nni + tyings.nnd)
        return A[u, u] + A[u, d] @ T + T.T @ A[d, u] + T.T @ A[d, d] @ T

    return mesh, vec, quad, K, G, tyings, dense


@pytest.mark.parametrize("size", [(10, 9), (32, 8), (5, 4, 6)])
@pytest.mark.parametrize("kind", ["merged", "spare"])
def test_cells_whose_unknowns_are_not_one_per_node(gf, size, kind):
    """A Regular cell in which unknowns of several nodes are one (rigid parts), and one with unknowns that no
    element uses: the product sums every node of an unknown, and is zero where there is none (1e-13: FP64 sums
    of some ten terms).  Such cells are no grid of unknowns, so the general operator takes them."""
    nd = len(size)
    merge = [(3 * nd, 3 * nd + nd, 3 * nd + 2 * nd), (1, 8 * nd + 1)] if kind == "merged" else []
    mesh, vec, quad, K, G, ty, dense = tied_cell(gf, size, merge, 2 if kind == "spare" else 0)
    P = gf.TyingsPCG(vec, quad, K, G, ty)
    A = dense(mesh.coor)
    rng = np.random.default_rng(3)
    for _ in range(2):  # the second product finds the first one's result in the pool
        xu = rng.standard_normal(ty.nnu)
        y = host(P.apply(xu))
        assert np.linalg.norm(y - A @ xu) <= 1e-13 * np.linalg.norm(A @ xu)
    assert not P.structured
    if kind == "merged":
        b = A @ xu
        x, _, res = P.solve(b, tol=1e-10)
        assert res <= 1e-9 and np.linalg.norm(b - A @ host(x)) <= 1e-9 * np.linalg.norm(b)


@pytest.mark.parametrize("size", [(10, 9), (32, 8), (5, 4, 6)])
def test_operator_follows_the_quadrature(gf, size):
    """update_x on the quadrature of an operator: products and solves are those of the coordinates in force,
    uneven ones (no shared geometry, so no structured kernel), even ones again, and stretched ones."""
    mesh, vec, quad, K, G, ty, dense = tied_cell(gf, size)
    P = gf.TyingsPCG(vec, quad, K, G, ty)
    assert P.structured
    nd = len(size)
    rng = np.random.default_rng(4)
    uneven = mesh.coor + 0.1 * np.sin(2.0 * np.pi * mesh.coor / np.array(size)[None, ::-1])
    for coor, even in ((mesh.coor, True), (uneven, False), (mesh.coor, True), (mesh.coor * (1.5, 0.75, 2.0)[:nd], True)):
        quad.update_x(oracle.Vector(mesh.conn, oracle.dofs(mesh.nnode, nd)).AsElement(coor))
        A = dense(coor)
        xu = rng.standard_normal(ty.nnu)
        y = host(P.apply(xu))
        assert np.linalg.norm(y - A @ xu) <= 1e-13 * np.linalg.norm(A @ xu)
        P.set_moduli(K, G)
        assert np.allclose(host(P.inverse_diagonal), 1.0 / np.diag(A), rtol=1e-13)
        b = A @ xu
        x, _, res = P.solve(b, tol=1e-10)
        assert res <= 1e-9 and np.linalg.norm(b - A @ host(x)) <= 1e-9 * np.linalg.norm(b)
        assert P.structured == even
        y = host(P.apply(xu))
        assert np.linalg.norm(y - A @ xu) <= 1e-13 * np.linalg.norm(A @ xu)
