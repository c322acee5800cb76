"""The reference-order FP64 step on either side of its dispatch: four lanes per element on grids of up to
2500 tiles of 15 x 3 nodes, one thread per element above.  Bit-exact with the oracle at the edges of the
tiles, with distorted coordinates, varying moduli, any mass and a force."""

import numpy as np
import pytest

import oracle
from oracle import QUAD4_PLANAR
from test_gpu_core import _explicit_setup, gf, host  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,distort,kvar,any_mass,force", [
    (1, 1, False, False, False, False), (13, 1, False, True, False, False), (14, 2, True, False, False, True),
    (15, 3, False, True, True, False), (16, 4, True, True, False, False), (28, 5, False, False, True, True),
    (29, 6, True, True, True, True), (30, 7, False, False, False, False), (44, 90, True, False, False, False),
    (374, 299, False, True, False, False),  # 25 x 100 = 2500 tiles: the last grid of this kernel
    (374, 300, False, True, False, False),  # 25 x 101
    (400, 330, True, False, True, True)])
def test_split_step_bit_exact(gf, nx, ny, distort, kvar, any_mass, force):  # noqa: F811
    coor, conn, dofs, q, inv, Ke, Ge, u, v, a = _explicit_setup(nx, ny, fixed=ny > 1, distort=distort, kvar=kvar)
    if any_mass:
        inv = inv * (1.0 + 0.2 * oracle.randn(77, inv.size))
    fext = 1e-3 * oracle.randn(5, inv.size) if force else None
    X = gf.ExplicitQuad4(gf.Vector(conn, dofs), coor, Ke, Ge, inv, 0.01, fext=fext)
    assert X.structured
    X.set_state(u, v, a)
    for nsteps in (1, 4):
        fint = oracle.vv_steps(nsteps, QUAD4_PLANAR, conn, dofs, q.dNx, q.dV(), Ke, Ge, inv, 0.01, u, v, a, fext=fext)
        X.step(nsteps, gf.F64, store_fint=True)
        gu, gv, ga = (host(t) for t in X.state())
        assert np.array_equal(gu, u) and np.array_equal(gv, v) and np.array_equal(ga, a)
        assert np.array_equal(host(X.fint()), fint)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("nx,ny", [(1, 1), (14, 16), (127, 2)])  # 8, 510 and 768 DOFs: around a workgroup's 512
def test_state_copies(gf, nx, ny, offset):  # noqa: F811
    import torch

    coor, conn, dofs, q, inv, Ke, Ge, u, v, a = _explicit_setup(nx, ny, fixed=False)
    X = gf.ExplicitQuad4(gf.Vector(conn, dofs), coor, Ke, Ge, inv, 0.01)
    rng = np.random.default_rng(nx)
    ref = [rng.standard_normal(dofs.size) for _ in range(3)]
    X.set_state(*ref)
    assert all(np.array_equal(host(t), r) for t, r in zip(X.state(), ref))
    n = dofs.size
    buf = torch.full((3, n + 3), np.nan, dtype=torch.float64, device="cuda")
    gf._call("gf_explicit_copy_state", X._h, *(gf._vp(buf[i, offset:].data_ptr()) for i in range(3)), gf._stream())
    got = host(buf)
    assert all(np.array_equal(got[i, offset:offset + n], ref[i]) for i in range(3))
    assert np.isnan(got[:, :offset]).all() and np.isnan(got[:, offset + n:]).all()


@pytest.mark.parametrize("n", [1383, 1385])  # 1,915,456 and 1,920,996 nodes: the last with patches of 208, the first of 256
def test_general_mesh_on_either_side_of_the_cache(gf, n):  # noqa: F811
    coor, conn, dofs, q, inv, Ke, Ge, u, v, a = _explicit_setup(n, n, shuffle=True)
    X = gf.ExplicitQuad4(gf.Vector(conn, dofs), coor, Ke, Ge, inv, 0.01)
    X.set_state(u, v, a)
    oracle.vv_steps(1, QUAD4_PLANAR, conn, dofs, q.dNx, q.dV(), Ke, Ge, inv, 0.01, u, v, a)
    X.step(1, gf.F64)
    assert all(np.array_equal(host(g), r) for g, r in zip(X.state(), (u, v, a)))
