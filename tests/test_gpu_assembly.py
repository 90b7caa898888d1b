"""GPU C0 assembly and matrix-free Helmholtz solve against the CPU checks of
tests/test_assembly_cpu.py (the same map, dense element matrices, scipy sparse solve)."""
import numpy as np
import pytest
import torch

import ithaca_hip as H
from ithaca_hip import assembly, mesh
import oracle as O
import os
import scipy.sparse as sp
import scipy.sparse.linalg as spla
import dense_ref as DR
from ithaca_hip import nektar_io as N
from test_assembly_cpu import _mesh, _qmesh, cpu_solve, l2_error, manufactured

pytestmark = pytest.mark.gpu


def _dev(a, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype=dtype)


def _gpu_problem(verts, ids, nm, nq, lam, dirichlet=True):
    E = len(ids)
    b = H.basis_modified_a(nm, nq)
    vd = _dev(verts)
    jac, df = H.geom_device("hex", vd, nq, b["z"], True)
    Hop = H.Operator("Helmholtz_Hex_Deformed", nm, nq, E, basis=b)
    Hop.set_jac(jac)
    Hop.set_df(df)
    Hop.set_lambda(lam)
    ipr = H.Operator("IProduct_Hex_Deformed", nm, nq, E, basis=b)
    ipr.set_jac(jac)
    u, f = manufactured(lam)
    X = mesh.hex_quad_points(vd, b["z"]).reshape(-1, 3)
    fx = ((3 * np.pi ** 2 + lam) * torch.sin(np.pi * X[:, 0]) * torch.sin(np.pi * X[:, 1])
          * torch.sin(np.pi * X[:, 2]))
    A = assembly.Assembly(ids, nm, dirichlet=dirichlet)
    rhs = A.assemble(ipr.apply(fx.contiguous()))
    return A, Hop, rhs, b


def test_gather_and_assemble_match_the_map():
    verts, ids = _mesh(3, True, seed=7, jitter=0.1)
    nm = 5
    l2g, sign, _, ng = assembly.assembly_map_hex(ids, nm)
    A = assembly.Assembly(ids, nm, dirichlet=False)
    assert A.nglobal == ng
    rng = np.random.default_rng(2)
    g = rng.uniform(-1, 1, ng)
    loc = A.global_to_local(_dev(g)).cpu().numpy()
    assert np.array_equal(loc, sign * g[l2g])
    lv = rng.uniform(-1, 1, len(l2g))
    ref = np.zeros(ng)
    np.add.at(ref, l2g, sign * lv)
    got = A.assemble(_dev(lv)).cpu().numpy()
    assert np.abs(got - ref).max() < 1e-13


@pytest.mark.parametrize("nm", [4, 6])
def test_helmsolve_matches_cpu_sparse_solve(nm):
    nq = nm + 1
    verts, ids = _mesh(2, True, seed=3, jitter=0.05)
    print(f"[case] helmsolve rotated 2^3 mesh nm={nm}", flush=True)
    x_cpu, l2g, sign, u = cpu_solve(verts, ids, nm, nq, 10.0)
    A, Hop, rhs, _ = _gpu_problem(verts, ids, nm, nq, 10.0)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-13, max_iter=5000)
    xg = x.cpu().numpy()
    print(f"iterations {it}, residual {res:.2e}")
    assert res < 1e-13
    assert np.linalg.norm(xg - x_cpu) <= 1e-9 * np.linalg.norm(x_cpu)
    e_gpu = l2_error(verts, ids, nm, nq, xg, l2g, sign, u)
    e_cpu = l2_error(verts, ids, nm, nq, x_cpu, l2g, sign, u)
    assert abs(e_gpu - e_cpu) <= 1e-6 * e_cpu


def test_helmsolve_neumann_residual():
    """Natural boundary conditions (lambda > 0: SPD): the returned x satisfies
    Assemble(H(GlobalToLocal(x))) = b to the requested tolerance."""
    verts, ids = _mesh(3, True, seed=11, jitter=0.1)
    A, Hop, rhs, _ = _gpu_problem(verts, ids, 5, 6, 2.0, dirichlet=False)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-11)
    y = A.assemble(Hop.apply(A.global_to_local(x)))
    rel = (torch.linalg.vector_norm(y - rhs) / torch.linalg.vector_norm(rhs)).item()
    print(f"iterations {it}, residual {res:.2e}, check {rel:.2e}")
    assert rel < 1e-10


def test_helmsolve_reports_non_convergence():
    verts, ids = _mesh(2, False)
    A, Hop, rhs, _ = _gpu_problem(verts, ids, 5, 6, 1.0)
    with pytest.raises(H.MFError, match="maximum number of iterations"):
        A.helmsolve(Hop, rhs, tol=1e-14, max_iter=2)


# ---------------------------------------------------------------- quadrilaterals

def _gpu_quad_problem(verts, ids, nm, nq, lam, deformed=True, dirichlet=True):
    E = len(ids)
    b = H.basis_modified_a(nm, nq)
    geo = "Deformed" if deformed else "Regular"
    jac, df = H.geom_device("quad", _dev(verts), nq, b["z"], deformed)
    Hop = H.Operator(f"Helmholtz_Quad_{geo}", nm, nq, E, basis=b)
    Hop.set_jac(jac)
    Hop.set_df(df)
    Hop.set_lambda(lam)
    ipr = H.Operator(f"IProduct_Quad_{geo}", nm, nq, E, basis=b)
    ipr.set_jac(jac)
    _, f = manufactured(lam, 2)
    fx = f(O.coords_quad(verts, nq, b["z"]).T)  # host points of the quadrature grid
    A = assembly.Assembly(ids, nm, dirichlet=dirichlet, shape="quad")
    rhs = A.assemble(ipr.apply(_dev(fx)))
    return A, Hop, rhs


def test_quad_gather_and_assemble_match_the_map():
    verts, ids = _qmesh(4, True, seed=7, jitter=0.1)
    nm = 6
    l2g, sign, _, ng = assembly.assembly_map_quad(ids, nm)
    A = assembly.Assembly(ids, nm, dirichlet=False, shape="quad")
    assert A.nglobal == ng and A.nlocal == len(ids) * nm * nm
    rng = np.random.default_rng(3)
    g = rng.uniform(-1, 1, ng)
    assert np.array_equal(A.global_to_local(_dev(g)).cpu().numpy(), sign * g[l2g])
    lv = rng.uniform(-1, 1, len(l2g))
    ref = np.zeros(ng)
    np.add.at(ref, l2g, sign * lv)
    assert np.abs(A.assemble(_dev(lv)).cpu().numpy() - ref).max() < 1e-13


@pytest.mark.parametrize("nm,deformed", [(5, True), (8, True), (5, False)])
def test_quad_helmsolve_matches_cpu_sparse_solve(nm, deformed):
    nq = nm + 1
    if deformed:
        verts, ids = _qmesh(4, True, seed=3, jitter=0.1)
    else:  # the regular 32x32 quads of the measured quad workload
        verts, ids = _qmesh(32, False)
    print(f"[case] quad helmsolve nm={nm} deformed={deformed} E={len(ids)}", flush=True)
    x_cpu, l2g, sign, u = cpu_solve(verts, ids, nm, nq, 1.0, "quad")
    A, Hop, rhs = _gpu_quad_problem(verts, ids, nm, nq, 1.0, deformed)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-13, max_iter=5000)
    xg = x.cpu().numpy()
    print(f"iterations {it}, residual {res:.2e}")
    assert res < 1e-13
    assert np.linalg.norm(xg - x_cpu) <= 1e-9 * np.linalg.norm(x_cpu)
    e_gpu = l2_error(verts, ids, nm, nq, xg, l2g, sign, u, "quad")
    e_cpu = l2_error(verts, ids, nm, nq, x_cpu, l2g, sign, u, "quad")
    # relative L2 errors; at nm = 8 they are ~3e-10, so allow round-off in absolute terms
    assert abs(e_gpu - e_cpu) <= 1e-6 * e_cpu + 1e-12


def test_quad_helmsolve_rejects_a_hex_operator():
    verts, ids = _qmesh(2, False)
    A = assembly.Assembly(ids, 4, shape="quad")
    b = H.basis_modified_a(4, 5)
    Hop = H.Operator("Helmholtz_Hex_Regular", 4, 5, len(ids), basis=b)
    rhs = torch.zeros(A.nglobal, dtype=torch.float64, device="cuda")
    with pytest.raises(H.MFError, match="Helmholtz operator"):
        A.helmsolve(Hop, rhs)


def test_smoothing_a_nektar_field():
    """The reference's FieldConvert Helmholtz smoother (ProcessC0Projection.cpp:196-224:
    lambda = (2 pi / L)^2 with L = 0.6, forcing -lambda u, natural boundary conditions) on
    the mesh and field of its test Hex_channel_C0helmsmoothing, through the GPU BwdTrans,
    IProduct, assembly and CG: the solution equals a dense-element sparse direct solve, and
    the seven printed L2 / "L inf" lines of Hex_channel_C0helmsmoothing.tst are reproduced
    at their tolerances.  As in the reference, the expansion comes from the field file
    (hexahedra: nm GLL points per direction, MeshGraph.cpp:1179-1183), the norms are taken
    after re-expanding on nm evenly spaced points per direction (OutputFileBase.cpp:83-86)
    and "L inf" is the largest signed value (ExpList.cpp:3034-3037)."""
    from test_nektar_io import SMOOTHING_GOLDEN, equispaced_rule, printed
    gold = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "nektar")
    nmesh = N.read_mesh(os.path.join(gold, "Hex_channel_C0helmsmoothing.xml"))
    blocks = N.read_fld(os.path.join(gold, "Hex_channel_C0helmsmoothing.fld"))
    lam = (2 * np.pi / 0.6) ** 2
    got = {}
    for f in ("u", "v", "w", "p"):
        print(f"[case] C0 Helmholtz smoothing of field {f}", flush=True)
        X, ids, c, nm, nq = N.expansion_arrays(nmesh, blocks, f, points="field")
        E, M = len(ids), nm ** 3
        # CPU: dense element matrices assembled with the same map, every mode free
        l2g, sign, _, ng = assembly.assembly_map_hex(ids, nm)
        rows, cols, vals, rhs = [], [], [], np.zeros(ng)
        for e in range(E):
            m = DR.element_mats("hex", nm, nq, X[e])
            g, s_ = l2g[e * M:(e + 1) * M], sign[e * M:(e + 1) * M].astype(float)
            rows.append(np.repeat(g, M))
            cols.append(np.tile(g, M))
            vals.append((DR.helmholtz_matrix(m, lam) * np.outer(s_, s_)).ravel())
            phys = m["B"] @ c[e * M:(e + 1) * M]
            np.add.at(rhs, g, s_ * (m["B"].T @ (m["W"] * m["J"] * lam * phys)))
        Ag = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))),
                           shape=(ng, ng))
        x_cpu = spla.spsolve(Ag.tocsc(), rhs)
        # GPU
        b = H.basis_modified_a(nm, nq)
        vd = _dev(X)
        jac, df = H.geom_device("hex", vd, nq, b["z"], True)
        Hop = H.Operator("Helmholtz_Hex_Deformed", nm, nq, E, basis=b)
        Hop.set_jac(jac)
        Hop.set_df(df)
        Hop.set_lambda(lam)
        ipr = H.Operator("IProduct_Hex_Deformed", nm, nq, E, basis=b)
        ipr.set_jac(jac)
        bwd = H.Operator("BwdTrans_Hex_Regular", nm, nq, E, basis=b)
        A = assembly.Assembly(ids, nm, dirichlet=False)
        phys = bwd.apply(_dev(c))
        x, it, res = A.helmsolve(Hop, A.assemble(ipr.apply(lam * phys)), tol=1e-13)
        print(f"iterations {it}, residual {res:.2e}")
        assert np.linalg.norm(x.cpu().numpy() - x_cpu) <= 1e-10 * np.linalg.norm(x_cpu)
        # the output expansion: nm evenly spaced points per direction, Newton-Cotes weights
        ze, we = equispaced_rule(nm)
        B1, _ = DR.modified_a(nm, ze)
        beq = dict(bdata=np.ascontiguousarray(B1.T.ravel()), dbdata=np.zeros(nm * nm),
                   D=np.zeros(nm * nm), w=we, nm=nm, nq=nm)
        out = H.Operator("BwdTrans_Hex_Regular", nm, nm, E, basis=beq)
        ue = out.apply(A.global_to_local(x))
        jeq, _ = H.geom_device("hex", vd, nm, ze, True)
        W = torch.from_numpy(np.kron(np.kron(we, we), we)).cuda()
        wj = (jeq.view(E, -1) * W).reshape(-1)
        got[f] = (torch.sqrt(torch.dot(wj * ue, ue)).item(), ue.max().item())
        if f == "u":
            Xe = mesh.hex_quad_points(vd, ze)
            for a, k in zip("xyz", range(3)):
                col = Xe[..., k].reshape(-1)
                got[a] = (torch.sqrt(torch.dot(wj * col, col)).item(), col.max().item())
    for name, l2, tl2, linf, tlinf in SMOOTHING_GOLDEN:
        print(f"{name}: L2 {got[name][0]:.7g} (golden {l2}), L inf {got[name][1]:.7g} "
              f"(golden {linf})")
        assert abs(printed(got[name][0]) - l2) <= tl2, name
        assert abs(printed(got[name][1]) - linf) <= tlinf, name


def test_helmholtz3d_hex_golden_on_the_gpu():
    """The reference's Demos/MultiRegions/Tests/Helmholtz3D_CG_Hex.tst (L2 error
    1.11818e-07, Linf 5.66374e-07, tolerance 1e-12) through the GPU path: geometry,
    IProduct of the forcing, assembly, the inhomogeneous Dirichlet lift and CG on the GPU,
    errors at the GLL points from the GPU BwdTrans."""
    gold = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "nektar")
    msh = N.read_mesh(os.path.join(gold, "Helmholtz3D_Hex_P6.xml"))
    X, ids = msh.element_coords(), msh.vertex_ids()
    nm = msh.expansions[0]["nummodes"]
    nq, E, lam = nm + 1, len(ids), 1.0
    uex = lambda P: np.sin(np.pi / 2 * P[:, 0]) * np.sin(np.pi / 2 * P[:, 1]) * np.sin(np.pi / 2 * P[:, 2])
    b = H.basis_modified_a(nm, nq)
    jac, df = H.geom_device("hex", _dev(X), nq, b["z"], True)
    Hop = H.Operator("Helmholtz_Hex_Deformed", nm, nq, E, basis=b)
    Hop.set_jac(jac)
    Hop.set_df(df)
    Hop.set_lambda(lam)
    ipr = H.Operator("IProduct_Hex_Deformed", nm, nq, E, basis=b)
    ipr.set_jac(jac)
    bwd = H.Operator("BwdTrans_Hex_Regular", nm, nq, E, basis=b)
    P = mesh.hex_quad_points(_dev(X), b["z"]).reshape(-1, 3).cpu().numpy()
    A = assembly.Assembly(ids, nm, dirichlet=True)
    rhs = A.assemble(ipr.apply(_dev((lam + 3 * np.pi ** 2 / 4) * uex(P))))
    g = assembly.dirichlet_lift(X, ids, nm, uex)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-14, max_iter=5000, lift=g)
    d = bwd.apply(A.global_to_local(x)).cpu().numpy() - uex(P)
    wq = np.einsum("k,j,i->kji", b["w"], b["w"], b["w"]).ravel()
    wj = jac.cpu().numpy() * np.tile(wq, E)
    l2, linf = np.sqrt(np.sum(wj * d * d)), np.abs(d).max()
    print(f"iterations {it}, residual {res:.1e}, L2 {l2:.6e}, Linf {linf:.6e}")
    assert abs(l2 - 1.11818e-07) <= 1e-12
    assert abs(linf - 5.66374e-07) <= 1e-12


def test_helmholtz3d_hex_allbcs_golden_on_the_gpu():
    """Demos/MultiRegions/Tests/Helmholtz3D_CG_Hex_AllBCs.tst (L2 0.000416575, Linf
    0.000871589, tolerance 1e-12 on the printed values) through the GPU path: Dirichlet on
    two regions (the mask of the Dirichlet faces' closure and their lift), Neumann on two
    and Robin on two (the face integrals on the right-hand side and the Robin trace matrix
    inside the GPU conjugate gradients)."""
    from test_assembly_cpu import _allbcs_problem, _printed
    msh, uex, bc = _allbcs_problem()
    X, ids = msh.element_coords(), msh.vertex_ids()
    nm = msh.expansions[0]["nummodes"]
    nq, E, lam = nm + 1, len(ids), 1.0
    print(f"[case] allbcs E={E} nm={nm}", flush=True)
    b = H.basis_modified_a(nm, nq)
    jac, df = H.geom_device("hex", _dev(X), nq, b["z"], True)
    Hop = H.Operator("Helmholtz_Hex_Deformed", nm, nq, E, basis=b)
    Hop.set_jac(jac)
    Hop.set_df(df)
    Hop.set_lambda(lam)
    ipr = H.Operator("IProduct_Hex_Deformed", nm, nq, E, basis=b)
    ipr.set_jac(jac)
    bwd = H.Operator("BwdTrans_Hex_Regular", nm, nq, E, basis=b)
    P = mesh.hex_quad_points(_dev(X), b["z"]).reshape(-1, 3).cpu().numpy()
    A = assembly.Assembly(ids, nm, dirichlet=True)
    g, dmask = assembly.dirichlet_lift_faces(X, ids, nm, uex, bc["dirichlet"])
    brhs, rr, rc, rv = assembly.boundary_terms(X, ids, nm, bc["neumann"], bc["robin"])
    A.set_dirichlet_mask(dmask)
    A.set_robin(rr, rc, rv)
    rhs = A.assemble(ipr.apply(_dev((lam + 3 * np.pi ** 2 / 4) * uex(P)))) + _dev(brhs)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-14, max_iter=5000, lift=g)
    d = bwd.apply(A.global_to_local(x)).cpu().numpy() - uex(P)
    wq = np.einsum("k,j,i->kji", b["w"], b["w"], b["w"]).ravel()
    wj = jac.cpu().numpy() * np.tile(wq, E)
    l2, linf = np.sqrt(np.sum(wj * d * d)), np.abs(d).max()
    print(f"iterations {it}, residual {res:.1e}, L2 {l2:.9e}, Linf {linf:.9e}")
    assert abs(_printed(l2) - 0.000416575) <= 1e-12
    assert abs(_printed(linf) - 0.000871589) <= 1e-12
    # removing the Robin matrix and the mask again restores the all-Dirichlet assembly
    A.set_robin([], [], [])
    A.set_dirichlet_mask(None)
    with pytest.raises(H.MFError):
        A.set_robin([0], [A.nglobal], [1.0])


# ---------------------------------------------------------------- variable order

def _runs(nmv):
    """(first, end, order) of each run of equal-order elements, in element order."""
    runs, e0 = [], 0
    for e in range(1, len(nmv) + 1):
        if e == len(nmv) or nmv[e] != nmv[e0]:
            runs.append((e0, e, int(nmv[e0])))
            e0 = e
    return runs


def _varp_gpu_problem(verts, ids, nmv, lam, shape):
    dim = 3 if shape == "hex" else 2
    S = "Hex" if shape == "hex" else "Quad"
    _, f = manufactured(lam, dim)
    ops, loc = [], []
    for e0, e1, nm in _runs(nmv):
        nq = nm + 1
        b = H.basis_modified_a(nm, nq)
        v = verts[e0:e1]
        jac, df = H.geom_device(shape, _dev(v), nq, b["z"], True)
        Hop = H.Operator(f"Helmholtz_{S}_Deformed", nm, nq, e1 - e0, basis=b)
        Hop.set_jac(jac)
        Hop.set_df(df)
        Hop.set_lambda(lam)
        ipr = H.Operator(f"IProduct_{S}_Deformed", nm, nq, e1 - e0, basis=b)
        ipr.set_jac(jac)
        pts = (O.coords_hex if shape == "hex" else O.coords_quad)(v, nq, b["z"]).T
        loc.append(ipr.apply(_dev(f(pts))))
        ops.append(Hop)
    A = assembly.Assembly(ids, nmv, dirichlet=True, shape=shape)
    return A, ops, A.assemble(torch.cat(loc).contiguous())


@pytest.mark.parametrize("shape", ["hex", "quad"])
def test_variable_order_gather_and_assemble(shape):
    from test_assembly_varp import _offsets  # noqa: F401  (same layout as the CPU tests)
    verts, ids = (_mesh if shape == "hex" else _qmesh)(3, True, seed=8, jitter=0.1)
    nmv = np.random.default_rng(9).integers(3, 7, len(ids))
    l2g, sign, _, ng = assembly.assembly_map(ids, nmv, shape)
    assert (sign == 0).any()
    A = assembly.Assembly(ids, nmv, dirichlet=False, shape=shape)
    assert A.nglobal == ng and A.nlocal == len(l2g)
    rng = np.random.default_rng(4)
    g = rng.uniform(-1, 1, ng)
    assert np.array_equal(A.global_to_local(_dev(g)).cpu().numpy(), sign * g[l2g])
    lv = rng.uniform(-1, 1, len(l2g))
    ref = np.zeros(ng)
    np.add.at(ref, l2g, sign * lv)
    assert np.abs(A.assemble(_dev(lv)).cpu().numpy() - ref).max() < 1e-13


@pytest.mark.parametrize("shape", ["hex", "quad"])
def test_variable_order_helmsolve_matches_cpu_sparse_solve(shape):
    from test_assembly_varp import varp_solve, varp_error
    if shape == "hex":
        verts, ids = _mesh(3, True, seed=3, jitter=0.05)
        nmv = np.repeat([4, 6, 5], 9)  # one order per z layer (elements are z-major)
    else:
        verts, ids = _qmesh(6, True, seed=3, jitter=0.05)
        nmv = np.repeat([3, 7, 5, 5, 8, 4], 6)  # one order per row
    print(f"[case] variable-order helmsolve {shape} orders {sorted(set(nmv.tolist()))}", flush=True)
    x_cpu, l2g, sign, u = varp_solve(verts, ids, nmv, 10.0, shape)
    A, ops, rhs = _varp_gpu_problem(verts, ids, nmv, 10.0, shape)
    x, it, res = A.helmsolve(ops, rhs, tol=1e-13, max_iter=5000)
    xg = x.cpu().numpy()
    print(f"operators {len(ops)}, iterations {it}, residual {res:.2e}")
    assert res < 1e-13
    assert np.linalg.norm(xg - x_cpu) <= 1e-9 * np.linalg.norm(x_cpu)
    e_gpu = varp_error(verts, ids, nmv, xg, l2g, sign, u, shape)
    e_cpu = varp_error(verts, ids, nmv, x_cpu, l2g, sign, u, shape)
    assert abs(e_gpu - e_cpu) <= 1e-6 * e_cpu


def test_variable_order_rejects_mismatched_operators():
    verts, ids = _mesh(2, False)
    nmv = np.repeat([4, 5], 4)
    A, ops, rhs = _varp_gpu_problem(verts, ids, nmv, 1.0, "hex")
    with pytest.raises(H.MFError, match="modes"):
        A.helmsolve(ops[::-1], rhs)
    with pytest.raises(H.MFError, match="cover"):
        A.helmsolve(ops[:1], rhs)


def test_preconditioner_follows_new_geometry():
    """Re-setting an operator's geometry rebuilds the cached assembled diagonal: the solve
    with the reused operator equals, bit for bit and in iterations, the solve with a fresh
    operator on the new geometry."""
    verts, ids = _mesh(2, True, seed=3, jitter=0.05)
    nm, nq = 5, 6
    A, Hop, rhs, b = _gpu_problem(verts, ids, nm, nq, 10.0)
    A.helmsolve(Hop, rhs, tol=1e-12)  # caches the diagonal of the first geometry
    verts2 = np.ascontiguousarray(verts * np.array([1.0, 2.0, 0.5]))
    jac2, df2 = H.geom_device("hex", _dev(verts2), nq, b["z"], True)
    Hop.set_jac(jac2)
    Hop.set_df(df2)
    x1, it1, _ = A.helmsolve(Hop, rhs, tol=1e-12)
    A2, Hop2, _, _ = _gpu_problem(verts2, ids, nm, nq, 10.0)
    x2, it2, _ = A2.helmsolve(Hop2, rhs, tol=1e-12)
    print(f"iterations {it1} / {it2}")
    assert it1 == it2
    assert torch.equal(x1, x2)


def test_preconditioner_follows_a_recreated_operator():
    """An operator destroyed and created again (its handle may land at the freed address)
    on new geometry with the same lambda: the cached assembled diagonal is keyed on a
    process-wide geometry id, so the reused assembly solves exactly as a fresh one."""
    import gc
    verts, ids = _mesh(2, True, seed=3, jitter=0.05)
    nm, nq = 5, 6
    A, Hop, rhs, b = _gpu_problem(verts, ids, nm, nq, 10.0)
    A.helmsolve(Hop, rhs, tol=1e-12)  # caches the diagonal of the first geometry
    for s in (0.5, 2.0):
        del Hop
        gc.collect()
        verts2 = np.ascontiguousarray(verts * np.array([1.0, s, 1.0]))
        jac2, df2 = H.geom_device("hex", _dev(verts2), nq, b["z"], True)
        Hop = H.Operator("Helmholtz_Hex_Deformed", nm, nq, len(ids), basis=b)
        Hop.set_jac(jac2)
        Hop.set_df(df2)
        Hop.set_lambda(10.0)
        x1, it1, _ = A.helmsolve(Hop, rhs, tol=1e-12)
        A2, Hop2, _, _ = _gpu_problem(verts2, ids, nm, nq, 10.0)
        x2, it2, _ = A2.helmsolve(Hop2, rhs, tol=1e-12)
        print(f"scale {s}: iterations {it1} / {it2}")
        assert it1 == it2
        assert torch.equal(x1, x2)


@pytest.mark.parametrize("nm,nq,lam", [(2, 4, 1.0), (4, 5, 10.0), (8, 9, 10.0), (7, 14, 2.0)])
def test_iteration_limit_at_and_around_convergence(nm, nq, lam):
    """Iterations are queued in groups ahead of the convergence test: the solve stops at the same
    iteration with any limit that allows it (x bit for bit the same), one short of it reports
    limit + 1 iterations as the reference does, and a zero right-hand side takes none."""
    verts, ids = _mesh(2, True, seed=4, jitter=0.05)
    print(f"[case] cg limits nm={nm} nq={nq}", flush=True)
    A, Hop, rhs, _ = _gpu_problem(verts, ids, nm, nq, lam)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-10)
    assert res <= 1e-10 and it >= 2
    for limit in (it - 1, it, it + 3, it + 9):
        y, jt, rs = A.helmsolve(Hop, rhs, tol=1e-10, max_iter=limit)
        assert jt == it and rs == res and torch.equal(x, y)
    for limit in {0, max(it - 2, 0)}:
        with pytest.raises(H.MFError, match="maximum number of iterations"):
            A.helmsolve(Hop, rhs, tol=1e-10, max_iter=limit)
    z, kt, _ = A.helmsolve(Hop, torch.zeros_like(rhs), tol=1e-10)
    assert kt == 0 and not z.any()


def _solve_raw(A, op, rhs, x, tol, max_iter):
    """The solver's C entry: (status, iterations, residual), also where the limit ends it."""
    import ctypes
    it, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
    L = H.lib()
    st = L.imf_helmsolve_cg_device(A._h, op._h, ctypes.c_void_p(rhs.data_ptr()), ctypes.c_void_p(x.data_ptr()),
                                   ctypes.c_double(tol), max_iter, ctypes.byref(it), ctypes.byref(res),
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return st, it.value, res.value


def _quad_problem(n, nm, nq, lam, deformed):
    verts, ids = _qmesh(n, True, 5)
    b = H.basis_modified_a(nm, nq)
    jac, df = H.geom_device("quad", _dev(verts), nq, b["z"], deformed)
    op = H.Operator(f"Helmholtz_Quad_{'Deformed' if deformed else 'Regular'}", nm, nq, len(ids), basis=b)
    op.set_jac(jac)
    op.set_df(df)
    op.set_lambda(lam)
    return assembly.Assembly(ids, nm, shape="quad"), op, ids


@pytest.mark.parametrize("shape,nm,nq", [("hex", 2, 4), ("hex", 4, 5), ("hex", 8, 9), ("hex", 6, 12),
                                         ("hex", 8, 16), ("quad", 3, 4), ("quad", 8, 16)])
@pytest.mark.parametrize("deformed", [False, True])
def test_first_iterates_pin_the_diagonal(shape, nm, nq, deformed):
    """x after one and two iterations of conjugate gradients with the diagonal of the assembled
    operator, the diagonal read off the operator applied to unit vectors: an entry of it that is
    wrong changes the first iterate's direction there.  Bar: 1e-11, some 1e3 roundings of sums of
    up to 4 096 terms.  A solve that the limit ends reports limit + 1 iterations."""
    print(f"[case] first iterates {shape} nm={nm} nq={nq} deformed={deformed}", flush=True)
    lam = 3.0
    if shape == "hex":
        verts, ids = _mesh(3 if nm == 2 else 2, True, seed=4, jitter=0.05)
        A, op, _, b = _gpu_problem(verts, ids, nm, nq, lam)
        if not deformed:
            jac, df = H.geom_device("hex", _dev(verts), nq, b["z"], False)
            op = H.Operator("Helmholtz_Hex_Regular", nm, nq, len(ids), basis=b)
            op.set_jac(jac)
            op.set_df(df)
            op.set_lambda(lam)
    else:
        A, op, ids = _quad_problem(3, nm, nq, lam, deformed)
    l2g, _, bnd, _ = assembly.assembly_map(ids, nm, shape)
    free = torch.ones(A.nglobal, dtype=torch.float64, device="cuda")
    free[torch.from_numpy(l2g[bnd.astype(bool)].astype(np.int64)).cuda()] = 0.0
    apply = lambda v: A.assemble(op.apply(A.global_to_local(v))) * free
    dinv = torch.zeros_like(free)
    for g in torch.nonzero(free).ravel().tolist():
        e = torch.zeros_like(free)
        e[g] = 1.0
        dinv[g] = 1.0 / apply(e)[g]
    rhs = torch.from_numpy(np.random.default_rng(1).standard_normal(A.nglobal)).cuda()
    x, r = torch.zeros_like(rhs), rhs * free
    w = dinv * r
    p = w.clone()
    rho = r @ w
    for k in (1, 2):
        Ap = apply(p)
        alpha = rho / (p @ Ap)
        x = x + alpha * p
        r = r - alpha * Ap
        got = torch.empty_like(rhs)
        st, it, _ = _solve_raw(A, op, rhs, got, 1e-14, k)
        assert st != 0 and it == k + 1
        assert float((got - x).norm()) <= 1e-11 * float(x.norm()), k
        w = dinv * r
        p, rho = w + (r @ w) / rho * p, r @ w
    st, it, _ = _solve_raw(A, op, rhs, torch.empty_like(rhs), 1e-14, 0)
    assert st != 0 and it == 1


def test_solves_of_few_iterations_cost_no_more_applies_than_they_need():
    """Iterations queued past the last one, and those of a solve that needs none, do not apply the
    operator: on a mesh where an apply is the larger part of an iteration, a zero right-hand side
    takes less time than four applies (nine were run once), on quads and anisotropic hexes."""
    import time
    A, op, _ = _quad_problem(400, 6, 7, 1.0, True)
    verts, ids = _mesh(20, False, seed=2, jitter=0.02)
    nms, nqs = (5, 6, 5), (6, 7, 6)
    tabs = [H.basis_modified_a(m, q) for m, q in zip(nms, nqs)]
    jac, df = H.geom_device("hex", _dev(verts), nqs, [t["z"] for t in tabs], True)
    hop = H.Operator("Helmholtz_Hex_Deformed", nms, nqs, len(ids), basis=tabs)
    hop.set_jac(jac)
    hop.set_df(df)
    hop.set_lambda(1.0)
    for a, o in ((A, op), (assembly.Assembly(ids, nms), hop)):
        zero, loc = torch.zeros(a.nglobal, dtype=torch.float64, device="cuda"), torch.ones(a.nlocal, dtype=torch.float64, device="cuda")
        out = torch.empty_like(loc)

        def best(f):
            t = []
            for _ in range(7):
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                f()
                torch.cuda.synchronize()
                t.append(time.perf_counter() - t0)
            return min(t[1:])
        one = best(lambda: [o.apply(loc, out) for _ in range(20)]) / 20
        none = best(lambda: a.helmsolve(o, zero, tol=1e-9))
        print(f"apply {one * 1e6:.0f} us, solve of none {none * 1e6:.0f} us")
        assert none < 4 * one + 60e-6  # and the vector passes, two of which read and write the mesh


def test_helmsolve_of_many_hexes_satisfies_the_operator():
    """4 096 elements of 4 modes and 6 points, beyond the count from which the gathered Helmholtz
    kernel packs elements into 256 threads: the plain operator on the solution gives the right-hand
    side back on the free modes (bar: twice the solver's own relative residual, whose norm this is)."""
    verts, ids = _mesh(16, True, seed=8, jitter=0.02)
    print("[case] helmsolve 16^3 nm=4 nq=6", flush=True)
    A, Hop, rhs, _ = _gpu_problem(verts, ids, 4, 6, 10.0)
    x, it, res = A.helmsolve(Hop, rhs, tol=1e-9)
    _, _, bnd, _ = assembly.assembly_map_hex(ids, 4)
    free = torch.ones(A.nglobal, dtype=torch.bool, device="cuda")
    l2g = assembly.assembly_map_hex(ids, 4)[0]
    free[torch.from_numpy(l2g[bnd.astype(bool)].astype(np.int64)).cuda()] = False
    r = (rhs - A.assemble(Hop.apply(A.global_to_local(x))))[free]
    assert res <= 1e-9 and float(r.norm()) <= 2e-9 * float(rhs.norm())
