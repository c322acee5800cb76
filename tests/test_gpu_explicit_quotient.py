"""The reference-order FP64 step forms the quotients of the inverse Jacobian from one reciprocal wherever the
mesh allows it: bit-exact with the oracle's divisions on random geometries, on Jacobians with zeros, on
scales on either side of that range (2^-200 to 2^200 for the determinant), and after an overflow."""

import numpy as np
import pytest

import oracle
from oracle import QUAD4_PLANAR
from test_gpu_core import gf, host  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


def run(gf, coor, conn, nsteps=2, overflow=None, seed=3):  # noqa: F811
    rng = np.random.default_rng(seed)
    size = np.abs(coor).max()
    dofs = oracle.dofs(coor.shape[0], 2)
    q = oracle.Quadrature(QUAD4_PLANAR, oracle.Vector(conn, dofs).AsElement(coor))
    n = conn.shape[0]
    K, G = rng.uniform(5, 10, n).astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32)
    inv = rng.uniform(0.5, 2.0, dofs.size)
    u, v, a = (1e-3 * size * rng.standard_normal(dofs.size) for _ in range(3))
    if overflow is not None:
        u[overflow] = 1e308
        u[overflow + 2] = -1e308
    X = gf.ExplicitQuad4(gf.Vector(conn, dofs), coor, K, G, inv, 0.01)
    X.set_state(u, v, a)
    fint = oracle.vv_steps(nsteps, QUAD4_PLANAR, conn, dofs, q.dNx, q.dV(), K, G, inv, 0.01, u, v, a)
    X.step(nsteps, gf.F64, store_fint=True)
    for got, ref in zip((*X.state(), X.fint()), (u, v, a, fint)):
        assert np.array_equal(host(got), ref, equal_nan=overflow is not None)
    return X


def mesh(kind):
    """One mesh for each kernel: a small and a large grid, renumbered elements."""
    c, conn = oracle.quad4_regular(*{"small": (37, 23), "large": (390, 310), "general": (61, 47)}[kind])
    if kind == "general":
        conn = conn[np.random.default_rng(0).permutation(conn.shape[0])]
    return c, conn


@pytest.mark.parametrize("kind", ["small", "large", "general"])
@pytest.mark.parametrize("form", ["plain", "rotated", "distorted"])
@pytest.mark.parametrize("power", [0, -99, -101, 99, 101])
def test_quotients(gf, kind, form, power):  # noqa: F811
    c, conn = mesh(kind)
    if form == "rotated":  # zeros on the Jacobian's diagonal
        c = np.stack((-c[:, 1], c[:, 0]), axis=1)
    if form == "distorted":
        c = c + 0.25 * np.random.default_rng(1).uniform(-1, 1, c.shape)
    X = run(gf, np.ldexp(c, power), conn)
    assert X.structured == (kind != "general")


@pytest.mark.parametrize("kind", ["small", "general"])
def test_after_an_overflow(gf, kind):  # noqa: F811
    c, conn = mesh(kind)
    run(gf, c, conn, nsteps=1, overflow=400)
