"""Quadrature and vector kernels at the sizes where their workgroups end: element counts around 64 (Quad4
points per workgroup / 4) and 16, rules from one point to more points than a workgroup has threads,
arrays that are not 16-byte aligned, renumbered and shared DOFs.  FP64 bit-exact with the oracle, FP32
equal to FP32 arithmetic in the kernels' order on the FP64 geometry rounded once."""

import numpy as np
import pytest

import oracle
from oracle import HEX8, QUAD4, QUAD4_PLANAR

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gf():
    import torch

    import goosefem_amd

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    goosefem_amd.lib()
    return goosefem_amd


def host(t):
    import torch

    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def unaligned(a):
    """A device copy of a whose first value lies 4 (FP32) or 8 (FP64) bytes past a 16-byte boundary."""
    import torch

    t = torch.empty(a.size + 2, dtype=torch.float32 if a.dtype == np.float32 else torch.float64, device="cuda")
    v = t[1 : a.size + 1].view(a.shape)
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    assert v.data_ptr() % 16 != 0
    return v


def elements(et, nelem, seed):
    """nelem distorted unit elements (no shared nodes): x [nelem, nne, ndim]."""
    rng = np.random.default_rng(seed)
    c, conn = oracle.quad4_regular(1, 1) if et != HEX8 else oracle.hex8_regular(1, 1, 1)
    x = c[conn[0]][None] + rng.uniform(-0.2, 0.2, (nelem,) + c[conn[0]].shape)
    return x + rng.integers(0, 50, (nelem, 1, 1))


def rule(nd, nip, seed=3):
    rng = np.random.default_rng(seed)
    return rng.uniform(-0.9, 0.9, (nip, nd)), rng.uniform(0.5, 1.5, nip)


CASES = [(et, n, nip) for et in (QUAD4, QUAD4_PLANAR) for n, nip in
         [(1, 4), (63, 4), (64, 4), (65, 4), (130, 4), (257, 1), (5, 3), (86, 3), (30, 9), (3, 256), (2, 257), (2, 300)]]
CASES += [(HEX8, n, nip) for n, nip in [(1, 8), (15, 8), (16, 8), (17, 8), (33, 8), (129, 1), (65, 2), (43, 3), (10, 27),
                                        (2, 128), (2, 129)]]


@pytest.mark.parametrize("et,nelem,nip", CASES)
def test_quadrature_shapes(gf, et, nelem, nip):
    import torch

    nd = 3 if et == HEX8 else 2
    x = elements(et, nelem, nelem + nip)
    xi, w = (None, None) if nip == (8 if et == HEX8 else 4) else rule(nd, nip)
    q = oracle.Quadrature(et, x, xi, w)
    cls = {QUAD4: gf.Element.Quad4.Quadrature, QUAD4_PLANAR: gf.Element.Quad4.QuadraturePlanar, HEX8: gf.Element.Hex8.Quadrature}[et]
    gq = cls(x, xi, w)
    rng = np.random.default_rng(7)
    ue = rng.standard_normal(x.shape)
    for arg in (ue, unaligned(ue)):
        for name in ("GradN_vector", "GradN_vector_T", "SymGradN_vector"):
            assert np.array_equal(host(getattr(gq, name)(arg)), getattr(q, name)(ue)), name
    out = unaligned(np.zeros((nelem, nip, gq.tdim, gq.tdim)))
    gq.SymGradN_vector(ue, out=out)
    assert np.array_equal(host(out), q.SymGradN_vector(ue))
    qt = rng.standard_normal((nelem, nip, gq.tdim, gq.tdim))
    ref = q.Int_gradN_dot_tensor2_dV(qt)
    assert np.array_equal(host(gq.Int_gradN_dot_tensor2_dV(qt)), ref)
    out = unaligned(np.zeros_like(ref))
    gq.Int_gradN_dot_tensor2_dV(unaligned(qt), out=out)
    assert np.array_equal(host(out), ref)
    # FP32, in the kernels' order
    g, v = q.GradN().astype(np.float32), q.dV().astype(np.float32)
    q32, u32 = qt.astype(np.float32), ue.astype(np.float32)
    f = np.zeros(x.shape, dtype=np.float32)
    for k in range(nip):
        a = g[:, k, :, 0, None] * q32[:, k, None, 0, :nd] + g[:, k, :, 1, None] * q32[:, k, None, 1, :nd]
        if nd == 3:
            a = a + g[:, k, :, 2, None] * q32[:, k, None, 2, :nd]
        f += a * v[:, k, None, None]
    assert np.array_equal(host(gq.Int_gradN_dot_tensor2_dV(torch.from_numpy(q32).cuda())), f)
    assert np.array_equal(host(gq.Int_gradN_dot_tensor2_dV(unaligned(q32))), f)
    e = np.zeros((nelem, nip, nd, nd), dtype=np.float32)
    for m in range(x.shape[1]):
        t = g[:, :, m, :, None] * u32[:, None, m, None, :]
        e = t if m == 0 and nd == 2 else e + t
    got = host(gq.GradN_vector(unaligned(u32)))
    assert np.array_equal(got[..., :nd, :nd], e) and not got[..., nd:, :].any() and not got[..., nd:].any()


@pytest.mark.parametrize("nelem,nip", [(1, 4), (63, 4), (64, 4), (65, 4), (200, 1), (29, 9), (17, 16), (43, 3)])
def test_axisymmetric_shapes(gf, nelem, nip):
    x = elements(QUAD4, nelem, nelem + nip)
    x[..., 1] += 3.0
    xi, w = (None, None) if nip == 4 else rule(2, nip)
    q = oracle.QuadratureAxisymmetric(x, xi, w)
    gq = gf.Element.Quad4.QuadratureAxisymmetric(x, xi, w)
    rng = np.random.default_rng(nip)
    ue, qt = rng.standard_normal(x.shape), rng.standard_normal((nelem, nip, 3, 3))
    for again in range(2):
        for name in ("GradN_vector", "GradN_vector_T", "SymGradN_vector"):
            assert np.array_equal(host(getattr(gq, name)(unaligned(ue))), getattr(q, name)(ue)), name
        ref = q.Int_gradN_dot_tensor2_dV(qt)
        out = unaligned(np.zeros_like(ref))
        gq.Int_gradN_dot_tensor2_dV(unaligned(qt), out=out)
        assert np.array_equal(host(out), ref) and np.array_equal(host(gq.Int_gradN_dot_tensor2_dV(qt)), ref)
        x = x + 0.05 * rng.standard_normal(x.shape)  # moved nodes are seen by every operator
        q.update_x(x)
        gq.update_x(x)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1000])
@pytest.mark.parametrize("td", [2, 3])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_elastic_stress_shapes(gf, n, td, dtype):
    import torch

    rng = np.random.default_rng(n)
    eps = rng.standard_normal((n, td, td)).astype(dtype)
    K, G = rng.uniform(1, 2, n).astype(dtype), rng.uniform(1, 2, n).astype(dtype)
    tr = (eps[:, 0, 0] + eps[:, 1, 1] + eps[:, 2, 2]) if td == 3 else eps[:, 0, 0] + eps[:, 1, 1]
    want = dtype(2) * G[:, None, None] * eps
    for i in range(td):
        want[:, i, i] = K * tr + dtype(2) * G * (eps[:, i, i] - tr / dtype(3))
    Kd, Gd = torch.from_numpy(K).cuda(), torch.from_numpy(G).cuda()
    assert np.array_equal(host(gf.elastic_stress(torch.from_numpy(eps).cuda(), Kd, Gd)), want)
    assert np.array_equal(host(gf.elastic_stress(unaligned(eps), unaligned(K), Gd)), want)


@pytest.mark.parametrize("numbering", ["identity", "permuted", "shared", "holes"])
@pytest.mark.parametrize("et", [QUAD4, HEX8])
def test_vector_numberings(gf, et, numbering):
    import torch

    rng = np.random.default_rng(1)
    c, conn = oracle.quad4_regular(17, 16) if et == QUAD4 else oracle.hex8_regular(7, 5, 4)
    conn = conn[rng.permutation(conn.shape[0])]
    nd = c.shape[1]
    dofs = oracle.dofs(c.shape[0], nd)
    if numbering == "permuted":
        dofs = rng.permutation(c.size).reshape(c.shape)
    elif numbering == "shared":  # as many numbers as entries would need, two nodes sharing one
        dofs[5] = dofs[11]
    elif numbering == "holes":
        dofs = oracle.dofs(c.shape[0], nd)
        dofs[dofs == 7] = 8
    ov, gv = oracle.Vector(conn, dofs), gf.Vector(conn, dofs)
    nv, ev = rng.standard_normal(c.shape), rng.standard_normal((conn.shape[0], conn.shape[1], nd))
    for a in (nv, unaligned(nv)):
        assert np.array_equal(host(gv.AsElement(a)), ov.AsElement(nv))
    out = unaligned(np.zeros_like(ev))
    gv.AsElement(nv, out=out)
    assert np.array_equal(host(out), ov.AsElement(nv))
    want_d, want_n = ov.AssembleDofs(ev), ov.AsNode(ov.AssembleDofs(ev))
    for a in (ev, unaligned(ev)):
        assert np.array_equal(host(gv.AssembleDofs(a)), want_d)
        assert np.array_equal(host(gv.AssembleNode(a)), want_n)
    e32 = ev.astype(np.float32)
    want_d = ov.AssembleDofs(e32.astype(np.float64))
    for a in (torch.from_numpy(e32).cuda(), unaligned(e32)):
        assert np.array_equal(host(gv.AssembleDofs(a)), want_d)
        assert np.array_equal(host(gv.AssembleNode(a)), ov.AsNode(want_d))


@pytest.mark.parametrize("nelem", [399999, 400000, 400007])
def test_hex8_fp32_integral_of_large_arrays(gf, nelem):
    """From 400,000 elements on the FP32 integral streams everything through LDS; the same bits as a few
    elements at a time."""
    import torch

    x = elements(HEX8, 500, 3)
    rng = np.random.default_rng(nelem)
    qt = torch.from_numpy(rng.standard_normal((500, 8, 3, 3)).astype(np.float32)).cuda()
    few = host(gf.Element.Hex8.Quadrature(x).Int_gradN_dot_tensor2_dV(qt))
    idx = torch.arange(nelem, device="cuda") % 500
    many = gf.Element.Hex8.Quadrature(torch.from_numpy(x).cuda()[idx].contiguous())
    got = many.Int_gradN_dot_tensor2_dV(qt[idx].contiguous())
    assert torch.equal(got, torch.from_numpy(few).cuda()[idx])
