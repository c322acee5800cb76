"""The work whose speed is measured: whole calls of this package, as a finite-element program makes them.

Six kinds of work, each over the range of sizes, element types and data types that programs use:

  explicit    velocity-Verlet steps of a Quad4 plane-strain body, then the state read back
  force       one force evaluation through the quadrature interface: nodal displacements -> strain ->
              elastic stress -> nodal forces -> acceleration (AsElement, SymGradN_vector,
              elastic_stress, Int_gradN_dot_tensor2_dV, AssembleNode, MatrixDiagonal.Solve)
  stiffness   element matrices from a tangent, the sparse matrix assembled, one product with it
  statics     one Newton iteration of a J2 plate: fused element pass, MatrixPartitioned, its solve
  tied        one Newton iteration of a periodic J2 cell: the same with tied degrees of freedom
  periodic    a periodic elastic cell solved matrix-free for one shear increment (TyingsPCG)
"""

import math

import numpy as np
import torch

import goosefem_amd as gf

DT = 0.01
PRECISION = {"f64": gf.F64, "f32": gf.F32, "f64_fast": gf.F64_FAST, "bf16x3": gf.BF16X3}


def listed():
    return [
        # a small dynamics run (the size of the reference's own example), read back every 20 steps:
        # launches and call overheads
        dict(name="explicit_small_f64", kind="explicit", mesh="regular", nx=64, ny=64, precision="f64", steps=20),
        # the headline: 8.4 million degrees of freedom in single-precision elements
        dict(name="explicit_large_f32", kind="explicit", mesh="regular", nx=2048, ny=2048, precision="f32", steps=50),
        # a mesh refined around a weak layer, in the default precision
        dict(name="explicit_finelayer_f64", kind="explicit", mesh="finelayer", nx=729, ny=900, nfine=700,
             precision="f64", steps=20),
        # one evaluation on a coarse mesh: nothing but launches
        dict(name="force_q4_small", kind="force", etype="q4planar", nx=41, ny=30, nz=0, dtype="f64"),
        # two million Quad4 elements, the reference's precision
        dict(name="force_q4_large", kind="force", etype="q4planar", nx=1500, ny=1333, nz=0, dtype="f64"),
        # a 3-D body in single precision, odd sizes
        dict(name="force_hex8_f32", kind="force", etype="hex8", nx=83, ny=71, nz=67, dtype="f32"),
        # a solid of revolution
        dict(name="force_axi", kind="force", etype="axi", nx=601, ny=499, nz=0, dtype="f64"),
        # 3-D stiffness, assembled and applied, in the reference's precision
        dict(name="stiffness_hex8_f64", kind="stiffness", etype="hex8", nx=47, ny=43, nz=41, dtype="f64"),
        # the same with single-precision tangents on the matrix cores
        dict(name="stiffness_hex8_bf16x3", kind="stiffness", etype="hex8", nx=72, ny=64, nz=60, dtype="bf16x3"),
        # a plate under shear: every Newton iteration of a quasi-static program
        dict(name="statics_q4", kind="statics", nx=128, ny=112),
        # the reference's periodic elasto-plastic example
        dict(name="tied_q4", kind="tied", nx=96, ny=96),
        # an elastic cell of a size nobody tuned for
        dict(name="periodic_q4", kind="periodic", etype="q4planar", nx=250, ny=250, nz=0),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["explicit", "force", "force", "stiffness", "stiffness", "statics", "tied", "periodic"])
    c = dict(kind=kind)
    if kind == "explicit":
        c["mesh"] = rng.choice(["regular", "finelayer"])
        c["precision"] = rng.choice(["f64", "f32", "f64_fast"])
        c["steps"] = rng.choice([5, 20, 50])
        if c["mesh"] == "regular":
            c["nx"] = _log(rng, 24, 1700)
            c["ny"] = max(8, int(c["nx"] * rng.uniform(0.5, 1.1)))
        else:
            c["nx"] = 27 * _log(rng, 2, 40)
            c["ny"] = int(c["nx"] * rng.uniform(0.6, 1.2))
            c["nfine"] = int(c["ny"] * rng.uniform(0.3, 0.8))
    elif kind == "force":
        c["etype"] = rng.choice(["q4planar", "q4", "hex8", "axi"])
        c["dtype"] = "f64" if c["etype"] == "axi" else rng.choice(["f64", "f32"])
        c["nx"] = _log(rng, 4, 72) if c["etype"] == "hex8" else _log(rng, 8, 1200)
        c["ny"] = max(3, int(c["nx"] * rng.uniform(0.6, 1.1)))
        c["nz"] = max(2, int(c["nx"] * rng.uniform(0.6, 1.1))) if c["etype"] == "hex8" else 0
    elif kind == "stiffness":
        c["etype"] = rng.choice(["q4planar", "hex8", "hex8", "axi"])
        c["dtype"] = rng.choice(["f64", "bf16x3"]) if c["etype"] == "hex8" else "f64"
        c["nx"] = _log(rng, 4, 56) if c["etype"] == "hex8" else _log(rng, 8, 500)
        c["ny"] = max(3, int(c["nx"] * rng.uniform(0.6, 1.1)))
        c["nz"] = max(2, int(c["nx"] * rng.uniform(0.6, 1.1))) if c["etype"] == "hex8" else 0
    elif kind == "statics":
        c["nx"] = _log(rng, 16, 144)
        c["ny"] = max(8, int(c["nx"] * rng.uniform(0.5, 1.0)))
    elif kind == "tied":
        c["nx"] = c["ny"] = _log(rng, 12, 112)
    else:
        c["etype"] = rng.choice(["q4planar", "q4planar", "hex8"])
        n = _log(rng, 16, 250) if c["etype"] == "q4planar" else _log(rng, 6, 30)
        c["nx"] = c["ny"] = n
        c["nz"] = n if c["etype"] == "hex8" else 0
    return c


# -------------------------------------------------------------------------------------------------
# inputs
# -------------------------------------------------------------------------------------------------


def _mesh(case):
    if case.get("mesh") == "finelayer":
        return gf.Mesh.Quad4.FineLayer(case["nx"], case["ny"], 1.0, case["nfine"])
    if case.get("etype") == "hex8":
        return gf.Mesh.Hex8.Regular(case["nx"], case["ny"], case["nz"])
    return gf.Mesh.Quad4.Regular(case["nx"], case["ny"])


def _rng(seed, what):
    return np.random.default_rng([int(seed), what])


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _class(etype):
    return {"q4planar": gf.Element.Quad4.QuadraturePlanar, "q4": gf.Element.Quad4.Quadrature,
            "axi": gf.Element.Quad4.QuadratureAxisymmetric, "hex8": gf.Element.Hex8.Quadrature}[etype]


def _coor(case, seed, coor):
    """Nodal coordinates of a body that was meshed, not ruled: every node moved by up to a tenth of an
    element; an axisymmetric body is a hollow cylinder (columns z, r) of inner radius 8."""
    x = coor + _rng(seed, 1).uniform(-0.1, 0.1, coor.shape)
    if case.get("etype") == "axi":
        x[:, 1] += 8.0
    return x


def _displacement(seed, coor):
    """A smooth displacement of about a per cent strain with a per mille of noise."""
    r = _rng(seed, 2)
    F = 0.01 * r.standard_normal((coor.shape[1], coor.shape[1]))
    size = coor.max(0) - coor.min(0)
    wave = np.sin(2.0 * math.pi * coor / size[None, :] + r.uniform(0.0, 6.0, coor.shape[1])[None, :])
    return coor @ F.T + 0.01 * wave + 1e-3 * r.standard_normal(coor.shape)


def _vector(seed, shape):
    """A nodal vector without the smoothness of a displacement, as an iterative solver multiplies."""
    return _rng(seed, 7).standard_normal(shape)


def _moduli(seed, shape):
    """Bulk and (log-normal) shear moduli, one value per entry."""
    r = _rng(seed, 3)
    return np.full(shape, 10.0), np.exp(0.3 * r.standard_normal(shape))


def _explicit_inputs(case, seed, mesh):
    nodes = mesh.nnode
    bottom, top = mesh.nodesBottomEdge, mesh.nodesTopEdge
    r = _rng(seed, 4)
    G = np.exp(0.3 * r.standard_normal(mesh.nelem)).astype(np.float32)
    K = np.full(mesh.nelem, 10.0, dtype=np.float32)
    u = 1e-3 * r.standard_normal((nodes, 2))
    v = np.zeros((nodes, 2))
    for edge in (bottom, top):
        u[edge] = 0.0
    v[top, 0] = 1e-4
    return K, G, u.ravel(), v.ravel(), np.concatenate((bottom, top))


def _plate_inputs(case, seed, ne):
    """J2 plate or cell: bulk modulus, log-normal shear modulus, yield stress and hardening per point."""
    r = _rng(seed, 5)
    G = np.exp(0.3 * r.standard_normal(ne))[:, None] * np.ones((1, 4))
    sy = 0.02 * np.exp(0.2 * r.standard_normal(ne))[:, None] * np.ones((1, 4))
    return 10.0, G, sy, 0.4


def prepare(case, seed):
    return {"explicit": _prepare_explicit, "force": _prepare_force, "stiffness": _prepare_stiffness,
            "statics": _prepare_statics, "tied": _prepare_tied, "periodic": _prepare_periodic}[case["kind"]](case, seed)


def _prepare_explicit(case, seed):
    mesh = _mesh(case)
    coor = mesh.coor
    vec = gf.Vector(mesh.conn, mesh.dofs)
    nodal = gf.Element.Quad4.QuadraturePlanar(vec.AsElement(coor), gf.Element.Quad4.Nodal.xi(), gf.Element.Quad4.Nodal.w())
    M = gf.MatrixDiagonal(vec, None)
    M.assemble(nodal.Int_N_scalar_NT_dV(torch.ones((mesh.nelem, 4), dtype=torch.float64, device="cuda")))
    inv = M.Solve(torch.ones(vec.ndof, dtype=torch.float64, device="cuda"))
    K, G, u, v, fixed = _explicit_inputs(case, seed, mesh)
    inv.view(-1, 2)[_dev(fixed)] = 0.0
    X = gf.ExplicitQuad4(vec, coor, K, G, inv, DT)
    X.set_state(u, v, np.zeros_like(u))
    return dict(case=case, X=X)


def _prepare_force(case, seed):
    mesh = _mesh(case)
    coor = _coor(case, seed, mesh.coor)
    vec = gf.Vector(mesh.conn, mesh.dofs)
    x = vec.AsElement(coor)
    cls = _class(case["etype"])
    elem = gf.Element.Hex8 if case["etype"] == "hex8" else gf.Element.Quad4
    nodal = cls(x, elem.Nodal.xi(), elem.Nodal.w())
    M = gf.MatrixDiagonal(vec, None)
    M.assemble(nodal.Int_N_scalar_NT_dV(torch.ones((mesh.nelem, nodal.nip), dtype=torch.float64, device="cuda")))
    quad = cls(x)
    K, G = _moduli(seed, (mesh.nelem, quad.nip))
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    return dict(case=case, vec=vec, quad=quad, M=M, u=_dev(_displacement(seed, coor)), K=_dev(K).to(dtype),
                G=_dev(G).to(dtype), dtype=dtype)


def _prepare_stiffness(case, seed):
    mesh = _mesh(case)
    coor = _coor(case, seed, mesh.coor)
    vec = gf.Vector(mesh.conn, mesh.dofs)
    quad = _class(case["etype"])(vec.AsElement(coor))
    K, G = _moduli(seed, (mesh.nelem, quad.nip))
    C = gf.elastic_tangent(K, _dev(G), dtype=torch.float32 if case["dtype"] == "bf16x3" else None)
    return dict(case=case, quad=quad, C=C, A=gf.Matrix(vec, None), u=_dev(_vector(seed, coor.shape)))


def _prepare_statics(case, seed):
    mesh = _mesh(case)
    dofs = mesh.dofs
    iip = np.concatenate((dofs[mesh.nodesBottomEdge].ravel(), dofs[mesh.nodesTopEdge].ravel()))
    vec = gf.VectorPartitioned(mesh.conn, dofs, iip)
    quad = gf.Element.Quad4.QuadraturePlanar(vec.AsElement(mesh.coor))
    K, G, sy, H = _plate_inputs(case, seed, mesh.nelem)
    mat = gf.LinearHardening(np.full((mesh.nelem, 4), K), G, sy, H)
    mat.increment()
    disp, du = _plate_displacement(seed, mesh.coor, case)
    return dict(case=case, vec=vec, quad=quad, mat=mat, A=gf.MatrixPartitioned(vec), disp=_dev(disp), du=_dev(du),
                solver=gf.MatrixPartitionedSolver())


def _plate_displacement(seed, coor, case):
    """The plate sheared by 2 %, with what the last iteration left to correct; the top edge moves on by
    0.1 %."""
    y = coor[:, 1] / case["ny"]
    disp = np.zeros_like(coor)
    disp[:, 0] = 0.02 * coor[:, 1]
    disp += 1e-4 * _rng(seed, 6).standard_normal(coor.shape) * ((y > 0.0) & (y < 1.0))[:, None]
    du = np.zeros_like(coor)
    du[y == 1.0, 0] = 0.001 * case["ny"]
    return disp, du


def _cell(mesh):
    control = gf.Tyings.Control(mesh.coor, mesh.dofs)
    iip = np.concatenate((control.controlDofs.ravel(), control.dofs[mesh.nodesOrigin].ravel()))
    ty = gf.Tyings.Periodic(control.coor, control.dofs, control.controlDofs, mesh.nodesPeriodic, iip)
    return control, ty


def _prepare_tied(case, seed):
    mesh = _mesh(case)
    control, ty = _cell(mesh)
    Cdu, Cdp, Cdi = ty.Cdu_csr, ty.Cdp_csr, ty.Cdi_csr
    vec = gf.VectorPartitionedTyings(mesh.conn, ty.dofs, Cdu, Cdp, Cdi)
    quad = gf.Element.Quad4.QuadraturePlanar(vec.AsElement(control.coor))
    K, G, sy, H = _plate_inputs(case, seed, mesh.nelem)
    mat = gf.LinearHardening(np.full((mesh.nelem, 4), K), G, sy, H)
    mat.increment()
    disp, du = _cell_displacement(seed, mesh.coor, case)
    return dict(case=case, vec=vec, quad=quad, mat=mat, A=gf.MatrixPartitionedTyings(mesh.conn, ty.dofs, Cdu, Cdp),
                disp=_dev(disp), du=_dev(du), solver=gf.MatrixPartitionedTyingsSolver(tol=1e-10))


def _wrap(nx, ny):
    """The periodic image (0 .. nx ny - 1) of each node of the grid."""
    iy, ix = np.meshgrid(np.arange(ny + 1), np.arange(nx + 1), indexing="ij")
    return ((iy % ny) * nx + ix % nx).ravel()


def _cell_displacement(seed, coor, case):
    """A cell sheared by 2 % with a periodic remainder (the origin fixed); the shear goes on by 0.1 %.
    The two rows at the end are the control nodes' (the macroscopic displacement gradient)."""
    nx, ny = case["nx"], case["ny"]
    w = 1e-4 * _rng(seed, 6).standard_normal((nx * ny, 2))
    w[0] = 0.0
    disp = np.zeros((coor.shape[0] + 2, 2))
    disp[:-2, 0] = 0.02 * coor[:, 1]
    disp[:-2] += w[_wrap(nx, ny)]
    disp[-2, 1] = 0.02
    du = np.zeros_like(disp)
    du[-2, 1] = 0.001
    return disp, du


def _prepare_periodic(case, seed):
    mesh = _mesh(case)
    control, ty = _cell(mesh)
    vec = gf.Vector(mesh.conn, ty.dofs)
    quad = _class(case["etype"])(gf.Vector(mesh.conn, mesh.dofs).AsElement(mesh.coor))
    K, G = _moduli(seed, mesh.nelem)
    xp = np.zeros(ty.nnp)
    xp[ty.control[0, 1] - ty.nnu] = 0.001
    return dict(case=case, vec=vec, quad=quad, pcg=gf.TyingsPCG(vec, quad, K, G, ty), xp=_dev(xp))


# -------------------------------------------------------------------------------------------------
# one pass
# -------------------------------------------------------------------------------------------------


def run(state):
    kind = state["case"]["kind"]
    if kind == "explicit":
        X, case = state["X"], state["case"]
        X.step(case["steps"], PRECISION[case["precision"]])
        return X.state()
    if kind == "force":
        vec, quad = state["vec"], state["quad"]
        eps = quad.SymGradN_vector(vec.AsElement(state["u"]).to(state["dtype"]))
        sig = gf.elastic_stress(eps, state["K"], state["G"])
        f = vec.AssembleNode(quad.Int_gradN_dot_tensor2_dV(sig))
        return eps, sig, f, state["M"].Solve(f)
    if kind == "stiffness":
        quad, A = state["quad"], state["A"]
        if state["case"]["dtype"] == "bf16x3":
            Ke = quad.Int_gradN_dot_tensor4_dot_gradNT_dV(state["C"], gf.BF16X3)
        else:
            Ke = quad.Int_gradN_dot_tensor4_dot_gradNT_dV(state["C"])
        A.assemble(Ke)
        return Ke, A.Dot(state["u"])
    if kind in ("statics", "tied"):
        vec, A = state["vec"], state["A"]
        fe, Ke = state["mat"].newton_q4(state["quad"], vec.AsElement(state["disp"]))
        A.assemble(Ke)
        f = vec.AssembleNode(fe)
        return Ke, f, state["solver"].Solve(A, -f, state["du"])
    pcg, xp = state["pcg"], state["xp"]
    x, _, _ = pcg.solve(-pcg.apply(None, xp))
    return state["vec"].AsNode(pcg.expand(x, xp))


# -------------------------------------------------------------------------------------------------
# what a pass cannot do without
# -------------------------------------------------------------------------------------------------


def _sizes(case):
    if case.get("etype") == "hex8":
        ne = case["nx"] * case["ny"] * case["nz"]
        return ne, (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1), 8, 3
    if case.get("mesh") == "finelayer":
        mesh = _mesh(case)
        return mesh.nelem, mesh.nnode, 4, 2
    return case["nx"] * case["ny"], (case["nx"] + 1) * (case["ny"] + 1), 4, 2


def work(case):
    """Bytes: each input (coordinates, connectivity, moduli, displacements, tangent) read once, each
    output written once; operations: the sums of the products of the method, per element and point."""
    ne, nn, nne, nd = _sizes(case)
    nip, K, ndof = nne, nne * nd, nd * nn
    mesh_bytes = 8 * ndof + 4 * nne * ne
    kind = case["kind"]
    if kind == "explicit":
        # per step u, v, a read and written, the inverse mass, coordinates, connectivity and shear
        # modulus read; the state read back
        per_step = 64 * ndof + 20 * ne
        return {"bytes": case["steps"] * per_step + 48 * ndof, "flops": case["steps"] * (300 * ne + 10 * ndof)}
    if kind == "force":
        size = 4 if case["dtype"] == "f32" else 8
        td2 = 4 if case["etype"] == "q4" else 9
        point = 2 * size + 2 * td2 * size
        return {"bytes": mesh_bytes + 8 * ndof + ne * nip * point + 3 * 8 * ndof,
                "flops": ne * nip * (60 * nne + 30)}
    if kind == "stiffness":
        size = 4 if case["dtype"] == "bf16x3" else 8
        used = {"q4planar": 16, "axi": 25, "hex8": 81}[case["etype"]]
        voigt = 6 if nd == 3 else 4
        return {"bytes": mesh_bytes + ne * nip * used * size + ne * K * K * size + 2 * 8 * ndof,
                "flops": ne * nip * 2 * voigt * K * (voigt + K)}
    if kind in ("statics", "tied"):
        # the element pass; the iterative solve has no such count (a direct one would read the matrix once)
        return {"bytes": mesh_bytes + 8 * ndof + ne * (4 * 4 * 8 + 4 * 80 + 4 * 80 + 64 + 512) + ne * 64 * 8 + 24 * ndof,
                "flops": ne * (4 * 200 + 4 * 2 * 4 * 8 * 12) + 36 * ndof}
    return {"bytes": mesh_bytes + 16 * ne + 16 * ndof, "flops": ne * 2 * K * K}


def tolerance(case):
    # about four times the largest error against exact() that any case of the kind showed
    kind = case["kind"]
    if kind == "explicit":
        # 64 bits: |x| eps in the derivatives of the shape functions, formed from coordinates of up to
        # some thousand elements; 32 bits: the element forces
        return {"rel": 2e-6 if case["precision"] == "f32" else 2e-12}
    if kind == "force":
        # the element's displacement differences: the displacement grows with the body's size, the
        # strain does not
        size = max(case["nx"], case["ny"], case["nz"])
        return {"rel": 1e-5 + 6e-7 * size if case["dtype"] == "f32" else 2e-12}
    if kind == "stiffness":
        return {"rel": 1.2e-5 if case["dtype"] == "bf16x3" else 5e-13}
    # solves stop at a residual of 1e-12 (statics) or 1e-10 of the right-hand side; the error of the
    # solution is that times what the conditioning of the scaled system adds
    return {"rel": 1e-11 if kind == "statics" else 2e-9}


# -------------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch and numpy
# -------------------------------------------------------------------------------------------------

_Q4 = np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], dtype=np.float64)
_H8 = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], dtype=np.float64)


def _shape(nd, nodal):
    """Shape functions [point, node] and their derivatives [point, node, dim] at the points."""
    s = _Q4 if nd == 2 else _H8
    xi = s if nodal else s / math.sqrt(3.0)
    f = 1.0 + s[None, :, :] * xi[:, None, :]
    N = np.prod(f, axis=2) / 2**nd
    dN = np.stack([s[None, :, d] * np.prod(np.delete(f, d, axis=2), axis=2) for d in range(nd)], axis=2) / 2**nd
    return torch.from_numpy(N).cuda(), torch.from_numpy(dN).cuda()


def _geometry(case, x, nodal=False):
    """N, dN/dx [element, point, node, dim], dV [element, point] and the points' radius (axisymmetric)."""
    nd = x.shape[2]
    N, dN = _shape(nd, nodal)
    # J[d][k] = d x_k / d xi_d
    J = [[(dN[None, :, :, d] * x[:, None, :, k]).sum(2) for k in range(nd)] for d in range(nd)]
    if nd == 2:
        det = J[0][0] * J[1][1] - J[0][1] * J[1][0]
        inv = [[J[1][1] / det, -J[0][1] / det], [-J[1][0] / det, J[0][0] / det]]
    else:
        def cof(i, j):
            a, b = [r for r in range(3) if r != i], [r for r in range(3) if r != j]
            return (-1) ** (i + j) * (J[a[0]][b[0]] * J[a[1]][b[1]] - J[a[0]][b[1]] * J[a[1]][b[0]])

        det = sum(J[0][j] * cof(0, j) for j in range(3))
        inv = [[cof(j, i) / det for j in range(3)] for i in range(3)]
    dNx = torch.stack([sum(inv[i][d][:, :, None] * dN[None, :, :, d] for d in range(nd)) for i in range(nd)], dim=3)
    r = None
    if case.get("etype") == "axi":
        r = (N[None] * x[:, None, :, 1]).sum(2)
        det = det * 2.0 * math.pi * r
    return N, dNx, det, r


def _blocks(ne):
    return [(a, min(ne, a + 60000)) for a in range(0, ne, 60000)]


def _strain(case, N, dNx, r, ue):
    """Strain [element, point, td, td]."""
    g = [[(dNx[..., i] * ue[:, None, :, j]).sum(2) for j in range(ue.shape[2])] for i in range(ue.shape[2])]
    td = 2 if case.get("etype") == "q4" else 3
    eps = torch.zeros(dNx.shape[:2] + (td, td), dtype=torch.float64, device="cuda")
    if case.get("etype") == "axi":  # (z, r) components; tensors in (r, theta, z) order
        eps[..., 0, 0] = g[1][1]
        eps[..., 1, 1] = (N[None] * ue[:, None, :, 1]).sum(2) / r
        eps[..., 2, 2] = g[0][0]
        eps[..., 0, 2] = eps[..., 2, 0] = 0.5 * (g[0][1] + g[1][0])
        return eps
    for i in range(ue.shape[2]):
        for j in range(ue.shape[2]):
            eps[..., i, j] = 0.5 * (g[i][j] + g[j][i])
    return eps


def _stress(eps, K, G):
    td = eps.shape[-1]
    eye = torch.eye(td, dtype=torch.float64, device="cuda")
    tr = torch.diagonal(eps, dim1=-2, dim2=-1).sum(-1)[..., None, None]
    return K[..., None, None] * tr * eye + 2.0 * G[..., None, None] * (eps - tr / 3.0 * eye)


def _rows(case, N, dNx, r):
    """B [element, point, node, dim, td, td]: strain = sum B u, as the sparse list of its entries."""
    if case.get("etype") == "axi":
        dr, dz, nr = dNx[..., 1], dNx[..., 0], N[None] / r[..., None]
        return [(1, 0, 0, dr), (1, 1, 1, nr), (0, 2, 2, dz), (0, 0, 2, dr), (1, 2, 0, dz)]
    nd = dNx.shape[3]
    return [(j, i, j, dNx[..., i]) for j in range(nd) for i in range(nd)]  # (component, row, column, factor)


def _force(case, N, dNx, r, dV, sig):
    fe = torch.zeros((dNx.shape[0], dNx.shape[2], dNx.shape[3]), dtype=torch.float64, device="cuda")
    for c, i, j, b in _rows(case, N, dNx, r):
        fe[:, :, c] += (b * (sig[..., i, j] * dV)[..., None]).sum(1)
    return fe


def _stiffness(case, N, dNx, r, dV, C):
    """Element matrices; C(i, j, k, l) is a function returning the entry per point, or None for zero."""
    e, _, m, nd = dNx.shape
    Ke = torch.zeros((e, m, nd, m, nd), dtype=torch.float64, device="cuda")
    rows = _rows(case, N, dNx, r)
    for c, i, j, b in rows:
        for d, k, l, h in rows:
            t = C(i, j, l, k)
            if t is None:
                continue
            t = t * dV
            for q in range(dNx.shape[1]):
                Ke[:, :, c, :, d] += (b[:, q] * t[:, q, None])[:, :, None] * h[:, q][:, None, :]
    return Ke.reshape(e, m * nd, m * nd)


def _elastic(K, G):
    def C(i, j, k, l):
        a = 1.0 if (i == j and k == l) else 0.0
        s = 0.5 * ((i == k) * (j == l) + (i == l) * (j == k)) - a / 3.0
        return None if a == 0.0 and s == 0.0 else K * a + 2.0 * G * s

    return C


def _assemble(conn, fe, nn):
    f = torch.zeros((nn, fe.shape[2]), dtype=torch.float64, device="cuda")
    return f.index_add_(0, conn.reshape(-1), fe.reshape(-1, fe.shape[2]))


def exact(case, seed):
    return {"explicit": _exact_explicit, "force": _exact_force, "stiffness": _exact_stiffness, "statics": _exact_newton,
            "tied": _exact_newton, "periodic": _exact_periodic}[case["kind"]](case, seed)


def _exact_explicit(case, seed):
    mesh = _mesh(case)
    if mesh.nelem * case["steps"] > 300_000_000:
        return None
    conn, coor = _dev(mesh.conn), _dev(mesh.coor)
    K, G, u, v, fixed = _explicit_inputs(case, seed, mesh)
    K, G = _dev(K).double(), _dev(G).double()
    u, v = _dev(u).view(-1, 2), _dev(v).view(-1, 2)
    inv = 1.0 / _lumped(case, conn, coor)
    inv[_dev(fixed)] = 0.0
    N, dNx, dV, _ = _geometry(case, coor[conn])
    a = torch.zeros_like(u)
    for _ in range(case["steps"]):
        u = u + DT * v + 0.5 * DT * DT * a
        eps = _strain(case, N, dNx, None, u[conn])
        fe = _force(case, N, dNx, None, dV, _stress(eps, K[:, None], G[:, None]))
        an = -inv * _assemble(conn, fe, mesh.nnode)
        v = v + 0.5 * DT * (a + an)
        a = an
    return u.reshape(-1), v.reshape(-1), a.reshape(-1)


def _lumped(case, conn, coor):
    _, _, dV, _ = _geometry(case, coor[conn], nodal=True)
    m = torch.zeros(coor.shape[0], dtype=torch.float64, device="cuda").index_add_(0, conn.reshape(-1), dV.reshape(-1))
    return m[:, None].expand(-1, coor.shape[1]).contiguous()


def _exact_force(case, seed):
    mesh = _mesh(case)
    coor_h = _coor(case, seed, mesh.coor)
    conn, coor = _dev(mesh.conn), _dev(coor_h)
    u = _dev(_displacement(seed, coor_h))
    K, G = (_dev(a) for a in _moduli(seed, (mesh.nelem, conn.shape[1])))
    if case["dtype"] == "f32":
        K, G = K.float().double(), G.float().double()
    eps, sig, fe = [], [], []
    for a, b in _blocks(mesh.nelem):
        N, dNx, dV, r = _geometry(case, coor[conn[a:b]])
        eps.append(_strain(case, N, dNx, r, u[conn[a:b]]))
        sig.append(_stress(eps[-1], K[a:b], G[a:b]))
        fe.append(_force(case, N, dNx, r, dV, sig[-1]))
    f = _assemble(conn, torch.cat(fe), mesh.nnode)
    return torch.cat(eps), torch.cat(sig), f, f / _lumped(case, conn, coor)


def _exact_stiffness(case, seed):
    mesh = _mesh(case)
    coor_h = _coor(case, seed, mesh.coor)
    conn, coor = _dev(mesh.conn), _dev(coor_h)
    u = _dev(_vector(seed, coor_h.shape))
    K, G = (_dev(a) for a in _moduli(seed, (mesh.nelem, conn.shape[1])))
    Ke, fe = [], []
    for a, b in _blocks(mesh.nelem):
        N, dNx, dV, r = _geometry(case, coor[conn[a:b]])
        Ke.append(_stiffness(case, N, dNx, r, dV, _elastic(K[a:b], G[a:b])))
        ue = u[conn[a:b]]
        fe.append((Ke[-1] * ue.reshape(b - a, 1, -1)).sum(2).reshape(ue.shape))
    return torch.cat(Ke), _assemble(conn, torch.cat(fe), mesh.nnode)


def _j2(eps, K, G, sy, H):
    """Stress and tangent (a function of the four indices) of J2 plasticity with linear hardening, no
    plastic history."""
    eye = torch.eye(3, dtype=torch.float64, device="cuda")
    tr = torch.diagonal(eps, dim1=-2, dim2=-1).sum(-1)
    s = 2.0 * G[..., None, None] * (eps - tr[..., None, None] / 3.0 * eye)
    ss = (s * s).sum((-2, -1))
    q = torch.sqrt(1.5 * ss)
    phi = q - sy
    plastic = phi > 0.0
    dg = torch.where(plastic, phi / (3.0 * G + H), torch.zeros_like(phi))
    qq = torch.where(plastic, q, torch.ones_like(q))
    f = 1.0 - 3.0 * G * dg / qq
    c = torch.where(plastic, 6.0 * G * G * (dg / qq - 1.0 / (3.0 * G + H)), torch.zeros_like(q))
    n = torch.where(plastic[..., None, None], s / torch.sqrt(ss).clamp_min(1e-300)[..., None, None], torch.zeros_like(s))
    sig = K * tr[..., None, None] * eye + f[..., None, None] * s

    def C(i, j, k, l):
        a = 1.0 if (i == j and k == l) else 0.0
        d = 0.5 * ((i == k) * (j == l) + (i == l) * (j == k)) - a / 3.0
        return K * a + 2.0 * G * f * d + c * n[..., i, j] * n[..., k, l]

    return sig, C


def _block_solve(rows, cols, vals, b, level):
    """x of A x = b for the symmetric matrix of the triplets, whose unknowns couple only within a level
    and with the next and the previous one, the first and the last being neighbours too: elimination
    level by level, the last one kept to the end."""
    nl = int(level.max()) + 1
    order = np.argsort(level, kind="stable")
    start = np.searchsorted(level[order], np.arange(nl + 1))
    place = np.empty(level.size, dtype=np.int64)
    place[order] = np.arange(level.size) - start[level[order]]
    size = np.diff(start)

    def block(i, j):
        sel = (level[rows] == i) & (level[cols] == j) if nl <= 3 else by[(i, j)]
        B = np.zeros((size[i], size[j]))
        np.add.at(B, (place[rows[sel]], place[cols[sel]]), vals[sel])
        return B

    by = {}
    if nl > 3:
        key = level[rows] * nl + level[cols]
        o = np.argsort(key, kind="stable")
        cut = np.concatenate(([0], np.flatnonzero(np.diff(key[o])) + 1, [key.size]))
        by = {(int(key[o[s]]) // nl, int(key[o[s]]) % nl): o[s:t] for s, t in zip(cut[:-1], cut[1:])}
    none = np.zeros(0, dtype=np.int64)
    if nl > 3:
        for i in range(nl):
            for j in range(nl):
                if abs(i - j) <= 1 or j == nl - 1:
                    by.setdefault((i, j), none)
    last = nl - 1
    D = [block(i, i) for i in range(nl)]
    U = [block(i, i + 1) for i in range(last)]
    W = [block(i, last) if i < last - 1 else None for i in range(last)]
    rhs = [b[order[start[i]:start[i + 1]]].copy() for i in range(nl)]
    keep = []
    for i in range(last):
        side = [U[i], rhs[i][:, None]] if W[i] is None else [U[i], W[i], rhs[i][:, None]]
        X = np.linalg.solve(D[i], np.concatenate(side, axis=1))
        XU, y = X[:, :size[i + 1]], X[:, -1]
        keep.append((XU, None if W[i] is None else X[:, size[i + 1]:-1], y))
        D[i + 1] -= U[i].T @ XU
        rhs[i + 1] -= U[i].T @ y
        if W[i] is not None:
            XW = keep[-1][1]
            if i + 1 < last - 1:
                W[i + 1] -= U[i].T @ XW
            else:
                U[i + 1] -= U[i].T @ XW
            D[last] -= W[i].T @ XW
            rhs[last] -= W[i].T @ y
    x = [None] * nl
    x[last] = np.linalg.solve(D[last], rhs[last])
    for i in range(last - 1, -1, -1):
        XU, XW, y = keep[i]
        x[i] = y - XU @ x[i + 1] - (0.0 if XW is None else XW @ x[last])
    out = np.empty_like(b)
    out[order] = np.concatenate(x)
    return out


def _solve_grid(number, level, Ke, rhs_nodes, known):
    """Displacements of the numbered nodes (the element-wise numbers in `number`, the rows of `level`),
    given the right-hand side and the known entries (NaN: unknown)."""
    nd = known.shape[1]
    dof = (number[:, :, None] * nd + np.arange(nd)).reshape(number.shape[0], -1)
    flat = known.ravel().copy()
    free = np.isnan(flat)
    at = np.cumsum(free) - 1
    b = rhs_nodes.ravel().copy()
    xk = np.where(free, 0.0, flat)
    np.add.at(b, dof.ravel(), -(Ke @ xk[dof][:, :, None])[:, :, 0].ravel())
    rows, cols = np.repeat(dof, dof.shape[1], axis=1).ravel(), np.tile(dof, (1, dof.shape[1])).ravel()
    sel = free[rows] & free[cols]
    x = _block_solve(at[rows[sel]], at[cols[sel]], Ke.ravel()[sel], b[free], np.repeat(level, nd)[free])
    flat[free] = x
    return flat.reshape(known.shape)


def _exact_newton(case, seed):
    mesh = _mesh(case)
    conn_h, coor = mesh.conn, mesh.coor
    conn = _dev(conn_h)
    tied = case["kind"] == "tied"
    disp, du = (_cell_displacement if tied else _plate_displacement)(seed, coor, case)
    K, G, sy, H = _plate_inputs(case, seed, mesh.nelem)
    N, dNx, dV, r = _geometry(case, _dev(coor)[conn])
    sig, C = _j2(_strain(case, N, dNx, r, _dev(disp)[conn]), K, _dev(G), _dev(sy), H)
    fe = _force(case, N, dNx, r, dV, sig)
    Ke = _stiffness(case, N, dNx, r, dV, C)
    f = _assemble(conn, fe, mesh.nnode)
    Ke_h, f_h = Ke.cpu().numpy(), f.cpu().numpy()
    if not tied:
        y = coor[:, 1]
        known = np.where(((y == 0.0) | (y == case["ny"]))[:, None], du, np.nan)
        x = _solve_grid(conn_h, np.rint(y).astype(np.int64), Ke_h, -f_h, known)
        return Ke, f, x
    x = _cell_solve(case, conn_h, coor, Ke_h, -f_h, du[-2:])
    # forces of tied nodes: the tied numbering keeps them apart, and the control nodes carry none
    return Ke, torch.cat((f, torch.zeros((2, 2), dtype=torch.float64, device="cuda"))), x


def _cell_solve(case, conn, coor, Ke, rhs, control):
    """Displacement of a periodic cell: the macroscopic gradient plus a periodic part, zero at the
    origin; the control nodes' rows at the end."""
    nd = coor.shape[1]
    n = [case["nx"], case["ny"], case.get("nz", 0)][:nd]
    i = np.rint(coor).astype(np.int64) % np.array(n)[None, :]
    image = i[:, 0] + n[0] * (i[:, 1] if nd == 2 else i[:, 1] + n[1] * i[:, 2])
    affine = coor @ control.T
    b = np.zeros((int(np.prod(n)), nd))
    np.add.at(b, image, rhs)
    fa = (Ke @ affine[conn].reshape(conn.shape[0], -1, 1))[:, :, 0]
    np.add.at(b, image[conn].ravel(), -fa.reshape(-1, nd))
    known = np.full(b.shape, np.nan)
    known[0] = 0.0
    level = np.arange(b.shape[0]) // (n[0] if nd == 2 else n[0] * n[1])
    w = _solve_grid(image[conn], level, Ke, b, known)
    return np.concatenate((affine + w[image], control))


def _exact_periodic(case, seed):
    if case["etype"] == "hex8" and case["nx"] > 14:
        return None
    mesh = _mesh(case)
    conn_h, coor = mesh.conn, mesh.coor
    K, G = (_dev(a)[:, None] for a in _moduli(seed, mesh.nelem))
    N, dNx, dV, r = _geometry(case, _dev(coor)[_dev(conn_h)])
    ones = torch.ones_like(dV)
    Ke = _stiffness(case, N, dNx, r, dV, _elastic(K * ones, G * ones)).cpu().numpy()
    control = np.zeros((coor.shape[1], coor.shape[1]))
    control[0, 1] = 0.001
    return _cell_solve(case, conn_h, coor, Ke, np.zeros_like(coor), control)
