"""The sparse matrix path at the sizes where its kernels change form, bit for bit against the oracle (the
same sums in the same order): the FP64 Hex8 stiffness (two, four or eight lane groups per element by the
number of elements, and element counts that leave a wave partly empty), and the product on a nodevec,
which reads and writes through the DOF numbering unless that is the identity."""

import numpy as np
import pytest

import oracle
from oracle import HEX8

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


@pytest.mark.parametrize("n", [(1, 1, 1), (5, 1, 1), (13, 15, 21), (16, 16, 16), (3, 43, 127), (5, 29, 113)])
def test_stiffness_hex8_of_any_number_of_elements(gf, n):
    c, conn = oracle.hex8_regular(*n)
    rng = np.random.default_rng(sum(n))
    c = c + 0.1 * rng.uniform(-1, 1, c.shape)
    x = oracle.Vector(conn, oracle.dofs(c.shape[0], 3)).AsElement(c)
    q = oracle.Quadrature(HEX8, x)
    C = rng.standard_normal((q.nelem, 8, 3, 3, 3, 3))
    got = host(gf.Element.Hex8.Quadrature(x).Int_gradN_dot_tensor4_dot_gradNT_dV(C, gf.F64))
    assert np.array_equal(got, q.Int_gradN_dot_tensor4_dot_gradNT_dV(C))


def fan(n):
    """n quadrilaterals around node 0: the longest row of the matrix has 2 (1 + 3 n) entries."""
    return np.array([[0, 1 + 3 * e, 2 + 3 * e, 3 + 3 * e] for e in range(n)])


@pytest.mark.parametrize("numbering", ["identity", "permuted", "tied"])
@pytest.mark.parametrize("mesh", ["quad4", "hex8", 15, 20, 40])
def test_dot_on_a_nodevec(gf, mesh, numbering):
    import torch

    nd = 2
    if mesh == "quad4":
        c, conn = oracle.quad4_regular(7, 5)
        nnode = c.shape[0]
    elif mesh == "hex8":
        c, conn = oracle.hex8_regular(5, 4, 3)
        nnode, nd = c.shape[0], 3
    else:
        conn = fan(mesh)
        nnode = 1 + 3 * mesh
    rng = np.random.default_rng(nnode)
    dofs = oracle.dofs(nnode, nd)
    if numbering == "permuted":
        dofs = rng.permutation(nnode * nd).reshape(nnode, nd)
    elif numbering == "tied":
        # three nodes, no two of one element, share their DOFs
        far = [1, nnode // 2 + 1, nnode - 1] if isinstance(mesh, str) else [1, 4, nnode - 3]
        dofs = dofs.copy()
        dofs[far] = dofs[far[0]]
        dofs = np.unique(dofs, return_inverse=True)[1].reshape(nnode, nd)
    vec = gf.Vector(conn, dofs)
    Ke = rng.standard_normal((conn.shape[0], conn.shape[1] * nd, conn.shape[1] * nd))
    A = gf.Matrix(vec, None)
    A.assemble(torch.from_numpy(Ke).cuda())
    x = rng.standard_normal((nnode, nd))
    last = np.zeros(dofs.max() + 1)
    for k, d in enumerate(dofs.ravel()):
        last[d] = x.ravel()[k]
    ref = oracle.csr_dot(*oracle.matrix_assemble(conn, dofs, Ke), last)[dofs]
    xd = torch.from_numpy(x).cuda()
    assert np.array_equal(host(A.Dot(xd)), ref)
    out = torch.full((nnode, nd), np.nan, dtype=torch.float64, device="cuda")
    A.Dot(xd, out)
    assert np.array_equal(host(out), ref)
    # the result over its operand, and shifted by one entry into it
    buf = torch.empty(nnode * nd + 1, dtype=torch.float64, device="cuda")
    for a, b in ((0, 0), (0, 1), (1, 0)):
        buf[a:a + nnode * nd] = xd.ravel()
        A.Dot(buf[a:a + nnode * nd].view(nnode, nd), buf[b:b + nnode * nd].view(nnode, nd))
        assert np.array_equal(host(buf[b:b + nnode * nd].view(nnode, nd)), ref)


@pytest.mark.parametrize("nelem,nip", [(1, 4), (63, 1), (64, 3), (65, 4), (130, 5), (7, 9), (3, 16)])
def test_axisymmetric_stiffness(gf, nelem, nip):
    """Workgroups of 64 elements, points four at a time; a general tensor, so that every slot pairing counts."""
    import torch

    rng = np.random.default_rng(nelem + nip)
    c, conn = oracle.quad4_regular(nelem, 1)
    zr = np.stack((c[:, 0], 0.5 + c[:, 1]), axis=1) + 0.1 * rng.uniform(-1, 1, c.shape)
    x = oracle.Vector(conn, oracle.dofs(c.shape[0], 2)).AsElement(zr)
    xi, w = rng.uniform(-0.9, 0.9, (nip, 2)), rng.uniform(0.5, 1.5, nip)
    oq = oracle.QuadratureAxisymmetric(x, xi, w)
    gq = gf.Element.Quad4.QuadratureAxisymmetric(x, xi, w)
    C = rng.standard_normal((nelem, nip, 3, 3, 3, 3))
    ref = oq.Int_gradN_dot_tensor4_dot_gradNT_dV(C)
    assert np.array_equal(host(gq.Int_gradN_dot_tensor4_dot_gradNT_dV(C)), ref)
    # arrays that are not 16-byte aligned
    cb = torch.zeros(C.size + 1, dtype=torch.float64, device="cuda")
    cb[1:] = torch.from_numpy(C.ravel()).cuda()
    out = torch.zeros(ref.size + 1, dtype=torch.float64, device="cuda")
    gq.Int_gradN_dot_tensor4_dot_gradNT_dV(cb[1:].view(C.shape), out=out[1:].view(ref.shape))
    assert out[0].item() == 0.0
    assert np.array_equal(host(out[1:].view(ref.shape)), ref)


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (2, 2, 1), (5, 1, 1), (17, 19, 23)])
def test_matrix_core_stiffness_of_any_number_of_elements(gf, n):
    """Four elements per workgroup, the last one partly filled.  An operand keeps its first two bf16 parts: the second is at most 2^-9 of it and what
    is left 2^-18, so a product of two loses 3 * 2^-18 (both remainders and the low parts' product); the 72
    sums and the rounding of the operands in FP32 add 77 * 2^-24, all relative to the sum of the terms'
    magnitudes."""
    import torch

    c, conn = oracle.hex8_regular(*n)
    rng = np.random.default_rng(sum(n))
    c = c + 0.1 * rng.uniform(-1, 1, c.shape)
    x = oracle.Vector(conn, oracle.dofs(c.shape[0], 3)).AsElement(c)
    q = oracle.Quadrature(HEX8, x)
    C = rng.standard_normal((q.nelem, 8, 3, 3, 3, 3)).astype(np.float32)
    gq = gf.Element.Hex8.Quadrature(x)
    ref = q.Int_gradN_dot_tensor4_dot_gradNT_dV(C.astype(np.float64))
    Cd = torch.from_numpy(C).cuda()
    k32 = host(gq.Int_gradN_dot_tensor4_dot_gradNT_dV(Cd, gf.BF16X3))
    g, ab = np.abs(q.dNx), np.zeros_like(ref)
    for k in range(8):
        t = np.einsum("eijkl,enl,e->eijnk", np.abs(C[:, k], dtype=np.float64), g[:, k], q.dV()[:, k])
        ab += np.einsum("emi,eijnk->emjnk", g[:, k], t).reshape(ref.shape)
    assert (np.abs(k32 - ref) <= (3 * 2.0**-18 + 77 * 2.0**-24) * ab).all()
    k64 = host(gq.Int_gradN_dot_tensor4_dot_gradNT_dV(Cd.double(), gf.BF16X3))
    assert np.array_equal(k64.astype(np.float32), k32)
    buf = torch.full((k32.size + 2,), np.nan, dtype=torch.float32, device="cuda")
    out = buf[1:-1].view(k32.shape)  # not 16-byte aligned
    gq.Int_gradN_dot_tensor4_dot_gradNT_dV(Cd, gf.BF16X3, out=out)
    assert np.array_equal(host(out), k32) and np.isnan(host(buf[[0, -1]])).all()
