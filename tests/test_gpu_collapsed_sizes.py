"""Operators of the collapsed shapes at the sizes where their kernels' tiles end (one element,
one less and one more than a tile of 16, one more than a workgroup's 64; 2 to 8 modes, so
1 to 18 column tiles), against the CPU oracle.  Bar: 1e-12 relative, as for the operators'
other parity tests (about 1e3 roundings of 1e-16 with condition 10)."""
import numpy as np
import pytest
import torch

import ithaca_hip as H
import oracle as O

pytestmark = pytest.mark.gpu

REG = {"tri": [[0, 0], [1, 0], [0, 1]],
       "tet": [[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]],
       "prism": [[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0.5, 0, 1], [0.5, 1, 1]],
       "pyr": [[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0.5, 0.5, 0.9]]}


def _basis(shape, nm, nq):
    if shape == "tri":
        return O.basis_tri(nm, nq)
    if shape == "tet":
        return O.basis_tet(nm, nq, nq - 1, nq - 1)
    return getattr(O, f"basis_{shape}")(nm, nq, nq - 1)


def _tables(shape, b):
    raw = {"tri": [1], "tet": [1, 2], "prism": [2], "pyr": [2]}[shape]
    return [dict(bdata=b[f"bdata{d}"], dbdata=b[f"dbdata{d}"], D=b[f"D{d}"],
                 w=b[f"w{d}_raw"] if d in raw else b[f"w{d}"]) for d in range(2 if shape == "tri" else 3)]


def _rel(a, r):
    return np.linalg.norm(a - r) / np.linalg.norm(r)


@pytest.mark.parametrize("E", [1, 15, 17, 65])
@pytest.mark.parametrize("nm,extra", [(2, 1), (3, 2), (5, 1), (6, 2), (8, 1)])
@pytest.mark.parametrize("deformed", [False, True])
@pytest.mark.parametrize("shape", ["tri", "tet", "prism", "pyr"])
def test_element_counts_and_orders(shape, deformed, nm, extra, E):
    print(f"[case] {shape} nm={nm} nq=+{extra} E={E} deformed={deformed}", flush=True)
    nq = nm + extra
    rng = np.random.default_rng(E + nm)
    R = np.array(REG[shape], dtype=float)
    jitter = 0.1 if deformed or shape in ("tri", "tet") else 0.0
    verts = np.stack([R * rng.uniform(0.5, 2.0) + jitter * rng.uniform(-1, 1, R.shape) for _ in range(E)])
    b = _basis(shape, nm, nq)
    jac, df = getattr(O, f"geom_{shape}")(verts, b, deformed)
    geo, cap = "Deformed" if deformed else "Regular", shape.capitalize()
    u, f = rng.uniform(-1, 1, E * b["M"]), rng.uniform(-1, 1, E * b["Q"])
    du, dfq = torch.from_numpy(u).cuda(), torch.from_numpy(f).cuda()

    def op(kind, g=geo):
        o = H.Operator(f"{kind}_{cap}_{g}", nm, tuple(b[f"nq{d}"] for d in range(R.shape[1])), E,
                       basis=_tables(shape, b))
        if o.needs_jac():
            o.set_jac(jac)
        if o.needs_df():
            o.set_df(df)
        return o

    bw, ip, hm = op("BwdTrans", "Regular"), op("IProduct"), op("Helmholtz")
    dim = R.shape[1]
    pd = op("PhysDeriv").apply(dfq).cpu().numpy()
    assert _rel(pd, np.concatenate(getattr(O, f"physderiv_{shape}")(b, E, deformed, df, f))) < 1e-12
    v = rng.uniform(-1, 1, (dim, E * b["Q"]))
    assert _rel(op("IProductWRTDerivBase").apply(torch.from_numpy(v.reshape(-1)).cuda()).cpu().numpy(),
                getattr(O, f"iprodderiv_{shape}")(b, E, deformed, jac, df, *([*v] if dim == 2 else [v]))) < 1e-12
    hm.set_lambda(2.5)
    Bu = getattr(O, f"bwdtrans_{shape}")(b, E, u)
    Pf = getattr(O, f"iproduct_{shape}")(b, E, deformed, jac, f)
    assert _rel(bw.apply(du).cpu().numpy(), Bu) < 1e-12
    assert _rel(ip.apply(dfq).cpu().numpy(), Pf) < 1e-12
    assert _rel(hm.apply(du).cpu().numpy(),
                getattr(O, f"helmholtz_{shape}")(b, E, deformed, jac, df, 2.5, u)) < 1e-12
    # transposes by their definition, element by element
    by = lambda a, n: a.reshape(E, n)
    Bt = bw.apply_transpose(dfq).cpu().numpy()
    Pt = ip.apply_transpose(du).cpu().numpy()
    scale = np.linalg.norm(u) * np.linalg.norm(f)
    assert np.abs((by(Bt, b["M"]) * by(u, b["M"])).sum(1) - (by(Bu, b["Q"]) * by(f, b["Q"])).sum(1)).max() < 1e-12 * scale
    assert np.abs((by(Pt, b["Q"]) * by(f, b["Q"])).sum(1) - (by(Pf, b["M"]) * by(u, b["M"])).sum(1)).max() < 1e-12 * scale


@pytest.mark.parametrize("shape", ["prism", "tet", "pyr"])
def test_dbdata_that_is_not_d_bdata_is_still_used(shape):
    """The kernels that apply D^T in place of dbdata only take tables where the two agree: with
    dbdata doubled, the stiffness part (lambda = 0) is exactly twice as large."""
    nm, E = 4, 9
    rng = np.random.default_rng(3)
    R = np.array(REG[shape], dtype=float)
    verts = np.stack([R + 0.1 * rng.uniform(-1, 1, R.shape) for _ in range(E)])
    b = _basis(shape, nm, nm + 1)
    jac, df = getattr(O, f"geom_{shape}")(verts, b, True)
    u = torch.from_numpy(rng.uniform(-1, 1, E * b["M"])).cuda()
    got = []
    for c in (1.0, 2.0):
        tabs = [dict(t, dbdata=c * t["dbdata"]) for t in _tables(shape, b)]
        o = H.Operator(f"Helmholtz_{shape.capitalize()}_Deformed", nm, tuple(b[f"nq{d}"] for d in range(3)),
                       E, basis=tabs)
        o.set_jac(jac)
        o.set_df(df)
        o.set_lambda(0.0)
        got.append(o.apply(u).cpu().numpy())
    assert _rel(got[1], 2.0 * got[0]) < 1e-12


@pytest.mark.parametrize("shape,kind,deformed,nm,extra,E", [
    ("tri", "BwdTrans", False, 5, 1, 6001), ("tet", "Helmholtz", False, 6, 1, 3743),
    ("tet", "Helmholtz", False, 8, 4, 319), ("tet", "IProduct", False, 5, 1, 4561),
    ("tet", "IProduct", True, 5, 1, 7745), ("pyr", "IProduct", False, 3, 1, 3507),
    ("prism", "IProduct", False, 2, 1, 3009), ("tet", "BwdTrans", False, 3, 1, 30005),
    ("tet", "BwdTrans", False, 5, 4, 1231), ("prism", "BwdTrans", False, 5, 8, 607),
    ("pyr", "IProduct", True, 4, 4, 5951), ("prism", "Helmholtz", False, 4, 1, 12811),
    ("tet", "IProduct", False, 8, 4, 3509)])
def test_large_element_counts_agree_with_small_ones(shape, kind, deformed, nm, extra, E):
    """Element counts just beyond those from which an operator takes dense products, with a ragged
    last tile: the first, some middle and the last elements equal those of an operator of 65
    elements, whose kernel is another one (checked against the oracle above).  Both directions
    (the transpose of one direction of a transform is the other's kernel)."""
    print(f"[case] {shape} {kind} nm={nm} nq=+{extra} E={E} deformed={deformed}", flush=True)
    nq = nm + extra
    rng = np.random.default_rng(E)
    R = np.array(REG[shape], dtype=float)
    jitter = 0.1 if deformed or shape in ("tri", "tet") else 0.0
    verts = R[None] * rng.uniform(0.5, 2.0, (E, 1, 1)) + jitter * rng.uniform(-1, 1, (E,) + R.shape)
    b = _basis(shape, nm, nq)
    nqs = tuple(b[f"nq{d}"] for d in range(R.shape[1]))
    geo = "Deformed" if deformed else "Regular"

    def op(v):
        n = len(v)
        o = H.Operator(f"{kind}_{shape.capitalize()}_{geo}", nm, nqs, n, basis=_tables(shape, b))
        jac, df = H.geom_device(shape, torch.from_numpy(v).cuda(), nqs, None, deformed)
        if o.needs_jac():
            o.set_jac(jac)
        if o.needs_df():
            o.set_df(df)
            o.set_lambda(2.5)
        return o
    big = op(verts)
    sizes = {"Helmholtz": (b["M"], b["M"]), "BwdTrans": (b["M"], b["Q"]), "IProduct": (b["Q"], b["M"])}[kind]
    for transpose in (False, True) if kind != "Helmholtz" else (False,):
        ni, no = sizes[::-1] if transpose else sizes
        x = torch.from_numpy(rng.uniform(-1, 1, (E, ni))).cuda()
        run = lambda o, v: (o.apply_transpose if transpose else o.apply)(v.reshape(-1).contiguous())
        y = run(big, x).reshape(E, no)
        for a in (0, E // 2, E - 65):
            part = run(op(verts[a:a + 65].copy()), x[a:a + 65]).reshape(65, no)
            assert _rel(y[a:a + 65].cpu().numpy(), part.cpu().numpy()) < 1e-12, (transpose, a)


@pytest.mark.parametrize("key,few", [("Helmholtz_Tet_Regular", 16), ("Helmholtz_Pyr_Regular", 16)])
def test_making_an_operator_with_dense_tables_takes_little_longer(key, few):
    """The tables are read off one run of the general kernel: an operator that takes dense products
    is made within 3.5 times the time of one that does not (it was six times)."""
    import time

    def best(E):
        H.Operator(key, 5, 6, E)
        t = []
        for _ in range(10):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            H.Operator(key, 5, 6, E, basis=basis)
            t.append(time.perf_counter() - t0)
        return min(t)
    basis = H.Operator(key, 5, 6, 1).basis
    small, large = best(few), best(40000)
    print(f"{key}: {small * 1e6:.0f} us, with tables {large * 1e6:.0f} us")
    assert large < 3.5 * small


@pytest.mark.parametrize("shape,nm,nq,E", [("tri", 4, 5, 130), ("tet", 4, 5, 70), ("tet", 7, 8, 70),
                                           ("prism", 5, 6, 70), ("pyr", 6, 7, 70), ("hex", 5, 6, 4003),
                                           ("hex", 6, 7, 70), ("hex", 8, 9, 1501), ("quad", 6, 7, 130)])
@pytest.mark.parametrize("deformed", [False, True])
def test_helmholtz_over_its_own_input(shape, nm, nq, E, deformed):
    """An element's coefficients are all read before any of its results is written, in every kernel
    that Helmholtz takes: out may be the input, bit for bit."""
    rng = np.random.default_rng(E + nm)
    R = {"hex": [[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]],
         "quad": [[0, 0], [1, 0], [1, 1], [0, 1]], **REG}[shape]
    R = np.array(R, dtype=float)
    jitter = 0.1 if deformed or shape in ("tri", "tet") else 0.0
    verts = R[None] * rng.uniform(0.5, 2.0, (E, 1, 1)) + jitter * rng.uniform(-1, 1, (E,) + R.shape)
    box = shape in ("hex", "quad")
    o = H.Operator(f"Helmholtz_{shape.capitalize()}_{'Deformed' if deformed else 'Regular'}", nm, nq, E)
    pts = nq if box else {"tri": (nq, nq - 1), "tet": (nq, nq - 1, nq - 1)}.get(shape, (nq, nq, nq - 1))
    jac, df = H.geom_device(shape, torch.from_numpy(verts).cuda(), pts,
                            H.basis_modified_a(nm, nq)["z"] if box else None, deformed)
    o.set_jac(jac)
    o.set_df(df)
    o.set_lambda(2.0)
    u = torch.from_numpy(rng.uniform(-1, 1, o.in_size)).cuda()
    want = o.apply(u)
    got = u.clone()
    o.apply(got, out=got)
    assert torch.equal(got, want)
