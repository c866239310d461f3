"""The calls whose time counts: what programs have this library do, through its public entry points.

Five flows, each the loop of a driver after its mesh, numbering and boundary conditions are in hand:

assemble     integrate_* and finish: every element integrated, the sparse matrix (and load vector) on the host.
             method "sort" is the default of the integrate functions; "reuse" is what a time or parameter loop uses.
solve        the heat driver: integrate_heat, the load vector, Jacobi-PCG with the boundary values, the solution.
coo          the drop-in for SysmatAssemblerSparse: a COO stream that a user's own weak form left on the host.
coo_device   the same for a stream that is already on the device, by the allocation-free entry point.
batch        many uneven problems assembled by one launch, and their matrices read back.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "elfel.jl_amd"))
import elfel_hip as eh  # noqa: E402
from elfel_hip import _lib as L  # noqa: E402

COO_DEVICE_MAX = 1 << 20  # entries that the allocation-free entry point takes


def listed():
    return [
        # a submatrix or a coarse mesh inside a loop that may not allocate: nothing but launches and waits
        dict(name="coo_device_16", flow="coo_device", nx=16, ny=16, layout="csr"),
        # the largest stream of that entry point, about a million entries
        dict(name="coo_device_241", flow="coo_device", nx=241, ny=241, layout="csc"),
        # a user's own weak form (two dofs a node) integrated on the host: six million entries handed over
        dict(name="coo_host_290", flow="coo", nx=290, ny=290, layout="csc"),
        # the heat test's own problem on its largest mesh, 100 x 100 triangles, to the solution
        dict(name="heat_t3_100_solve", flow="solve", fe="T3", nx=100, ny=100, method="sort", precision="fp64"),
        # heat with a random conductivity on two million quadrilaterals, solved in mixed precision
        dict(name="heat_q4_1500_solve", flow="solve", fe="Q4", nx=1500, ny=1300, method="reuse", precision="mixed"),
        # one step of a parameter loop: new conductivities and sources, the matrix and the load read back
        dict(name="heat_q4_701_reuse", flow="assemble", form="heat", fe="Q4", nx=701, ny=523, nz=0, method="reuse",
             precision="mixed"),
        # elasticity by the defaults: a matrix for a direct solver on the host
        dict(name="elasticity_t6_200", flow="assemble", form="elasticity", fe="T6", nx=200, ny=200, nz=0, method="sort",
             precision="fp64"),
        # the benchmark's elasticity mesh, 320 000 quadratic triangles, with new stiffness scales
        dict(name="elasticity_t6_400_reuse", flow="assemble", form="elasticity", fe="T6", nx=400, ny=400, nz=0,
             method="reuse", precision="mixed"),
        # a Taylor-Hood system of an odd size, read back for an indefinite solver
        dict(name="stokes_t6t3_153_reuse", flow="assemble", form="stokes", fe="T6", nx=153, ny=149, nz=0, method="reuse",
             precision="fp64"),
        # a bubble / linear triangle pair in three scalar spaces, as the colliding-flow driver assembles it
        dict(name="reddy_p1b_131", flow="assemble", form="reddy", fe="T3B", nx=131, ny=127, nz=0, method="sort",
             precision="fp64"),
        # heat in three dimensions, the tetrahedra of the poisson driver
        dict(name="heat_t4_36", flow="assemble", form="heat", fe="T4", nx=36, ny=35, nz=37, method="sort", precision="fp64"),
        # twelve heat and elasticity problems of uneven size in one launch
        dict(name="batch_12", flow="batch", problems=12, emin=1000, emax=40000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, n):
    return max(2, int(round(n * rng.uniform(0.8, 1.0))))


def draw(rng):
    """One more case: the flow, then a size over the logarithm of its range."""
    kind = rng.choice(["coo_device", "coo", "solve_fp64", "solve_mixed", "heat2d", "elasticity", "stokes", "reddy",
                       "heat3d", "batch"])
    both = rng.choice([("sort", "fp64"), ("reuse", "fp64"), ("reuse", "mixed")])
    if kind == "coo_device":
        n = _log_int(rng, 12, 241)
        return dict(flow="coo_device", nx=n, ny=_near(rng, n), layout=rng.choice(["csr", "csc"]))
    if kind == "coo":
        n = _log_int(rng, 20, 290)
        return dict(flow="coo", nx=n, ny=_near(rng, n), layout=rng.choice(["csr", "csc"]))
    if kind == "solve_fp64":
        n = _log_int(rng, 40, 300)
        return dict(flow="solve", fe=rng.choice(["T3", "Q4"]), nx=n, ny=_near(rng, n), method=rng.choice(["sort", "reuse"]),
                    precision="fp64")
    if kind == "solve_mixed":
        n = _log_int(rng, 100, 1400)
        return dict(flow="solve", fe=rng.choice(["T3", "Q4"]), nx=n, ny=_near(rng, n), method="reuse", precision="mixed")
    if kind == "batch":
        return dict(flow="batch", problems=rng.randint(6, 14), emin=_log_int(rng, 500, 3000), emax=_log_int(rng, 8000, 40000))
    form, fe, lo, hi = {"heat2d": ("heat", rng.choice(["T3", "Q4"]), 20, 900), "elasticity": ("elasticity", "T6", 16, 380),
                        "stokes": ("stokes", "T6", 16, 250), "reddy": ("reddy", rng.choice(["T3B", "Q4"]), 20, 250),
                        "heat3d": ("heat", "T4", 6, 48)}[kind]
    if form == "reddy":
        both = ("sort", "fp64")
    n = _log_int(rng, lo, hi)
    return dict(flow="assemble", form=form, fe=fe, nx=n, ny=_near(rng, n), nz=_near(rng, n) if fe == "T4" else 0,
                method=both[0], precision=both[1])


# ---- the inputs ----------------------------------------------------------------
@functools.lru_cache(maxsize=8)
def _block(fe, nx, ny, nz):
    """Connectivity, node coordinates and boundary nodes of a block of cells, the unit square or cube."""
    if fe == "T4":
        m = eh.T4block(1.0, 1.0, 1.0, nx, ny, nz)
        b = np.nonzero(np.any((m.xy < 1e-12) | (m.xy > 1 - 1e-12), axis=1))[0] + 1
    else:
        m = {"T3": eh.T3block, "T3B": eh.T3block, "T6": eh.T6block, "Q4": eh.Q4block}[fe](1.0, 1.0, nx, ny)
        b = np.nonzero(np.any((m.xy < 1e-12) | (m.xy > 1 - 1e-12), axis=1))[0] + 1
    return m.conn, m.xy, b, m.shape


@functools.lru_cache(maxsize=4)
def _corners(nx, ny):
    m = eh.T6toT3(eh.Mesh(*(_block("T6", nx, ny, 0)[k] for k in (0, 1, 3))))
    return m.conn, m.xy


def _mesh(fe, nx, ny, nz, rng):
    """A block mesh with its inner nodes moved by up to a tenth of a cell."""
    conn, xy, b, shape = _block(fe, nx, ny, nz)
    d = rng.uniform(-0.1, 0.1, xy.shape) / max(nx, ny, nz)
    d[b - 1] = 0.0
    return eh.Mesh(conn, xy + d, shape), b


_FE = {"T3": eh.FEH1_T3, "T6": eh.FEH1_T6, "Q4": eh.FEH1_Q4, "T4": eh.FEH1_T4, "T3B": eh.FEH1_T3_BUBBLE}
_RULE = {"T3": dict(kind="default", npts=1), "T6": dict(kind="default", npts=3), "Q4": dict(kind="Gauss", order=2),
         "T4": dict(kind="default", npts=1), "T3B": dict(kind="default", npts=3)}


def _heat(case, rng):
    """Mesh, space, conductivity and source of a heat problem; boundary values 1 + x^2 + 2 y^2."""
    fe = case["fe"]
    mesh, b = _mesh(fe, case["nx"], case["ny"], case.get("nz", 0), rng)
    fesp = eh.FESpace(mesh, _FE[fe]())
    x = mesh.xy[b - 1]
    fesp.setebc(0, b, 1, 1.0 + x[:, 0] ** 2 + 2.0 * x[:, 1] ** 2)
    eh.numberdofs(fesp)
    p = dict(fesp=fesp, rule=_RULE[fe], kappa=float(rng.uniform(0.5, 2.0)), Q=float(rng.uniform(-6.0, -3.0)), kappa_e=None,
             Q_e=None)
    if fe == "Q4":
        p["kappa_e"] = np.exp(rng.standard_normal(mesh.nelements))
        p["Q_e"] = rng.uniform(-1.0, 1.0, mesh.nelements)
    return p


def _elasticity(case, rng):
    mesh, _ = _mesh("T6", case["nx"], case["ny"], 0, rng)
    fesp = eh.FESpace(mesh, eh.FEH1_T6(), 2)
    left = np.nonzero(mesh.xy[:, 0] < 1e-12)[0] + 1
    for c in (1, 2):
        fesp.setebc(0, left, c, 0.0)
    eh.numberdofs(fesp)
    return dict(fesp=fesp, rule=_RULE["T6"], D=eh.plane_strain_D(1.0, 0.3),
                scale_e=np.exp(0.5 * rng.standard_normal(mesh.nelements)))


def _stokes(case, rng):
    mesh, b = _mesh("T6", case["nx"], case["ny"], 0, rng)
    pconn, _ = _corners(case["nx"], case["ny"])
    pmesh = eh.Mesh(pconn, mesh.xy[: (case["nx"] + 1) * (case["ny"] + 1)], "T3")
    u = eh.FESpace(mesh, eh.FEH1_T6(), 2)
    for c in (1, 2):
        u.setebc(0, b, c, 0.0)
    p = eh.FESpace(pmesh, eh.FEH1_T3(), 1)
    p.setebc(0, pmesh.nearestto([0.5, 0.5]), 1, 0.0)
    eh.numberdofs([u, p])
    return dict(u=u, p=p, rule=_RULE["T6"], mu=float(rng.uniform(0.5, 2.0)))


def _reddy(case, rng):
    fe = case["fe"]
    mesh, b = _mesh(fe, case["nx"], case["ny"], 0, rng)
    ux, uy = eh.FESpace(mesh, _FE[fe]()), eh.FESpace(mesh, _FE[fe]())
    for s in (ux, uy):
        s.setebc(0, b, 1, 0.0)
    p = eh.FESpace(mesh, eh.FEL2_Q4() if fe == "Q4" else eh.FEH1_T3())
    p.setebc(2 if fe == "Q4" else 0, 1, 1, 0.0)
    eh.numberdofs([ux, uy, p])
    return dict(ux=ux, uy=uy, p=p, rule=_RULE[fe], mu=float(rng.uniform(0.5, 2.0)))


def _coo(case, rng):
    """The stream of an element loop over triangles, one or two dofs a node, the values of an element correlated."""
    nc = 2 if case["flow"] == "coo" else 1
    conn, xy, _, _ = _block("T3", case["nx"], case["ny"], 0)
    d = (np.repeat(conn - 1, nc, axis=1) * nc + np.tile(np.arange(nc), 3) + 1).astype(np.int64)
    nd = d.shape[1]
    I = np.tile(d, (1, nd)).ravel()
    J = np.repeat(d, nd, axis=1).ravel()
    V = rng.standard_normal(I.size) + np.repeat(rng.standard_normal(d.shape[0]), nd * nd)
    n = xy.shape[0] * nc
    if nc == 1 and I.size > COO_DEVICE_MAX:
        raise ValueError("more entries than the allocation-free entry point takes")
    return I, J, V, n


def _batch(case, rng):
    """Heat on triangles and quadrilaterals and elasticity in turn, of emin to emax elements in mixed order."""
    out = []
    for k in range(case["problems"]):
        e = case["emin"] * (case["emax"] / case["emin"]) ** ((0.618 * (k + 1)) % 1.0)
        kind = ("heat_t3", "elasticity", "heat_q4")[k % 3]
        n = max(2, int(round(math.sqrt(e if kind == "heat_q4" else e / 2))))
        sub = dict(nx=n, ny=max(2, n - 1), nz=0)
        if kind == "elasticity":
            p = _elasticity(sub, rng)
            coef = p["scale_e"]
        else:
            p = _heat(dict(sub, fe="T3" if kind == "heat_t3" else "Q4"), rng)
            coef = np.exp(0.5 * rng.standard_normal(p["fesp"].mesh.nelements))
        out.append((kind, p, coef))
    return out


_SETUP = {"heat": _heat, "elasticity": _elasticity, "stokes": _stokes, "reddy": _reddy}


def prepare(case, seed):
    rng = np.random.default_rng([seed, 1])
    flow = case["flow"]
    s = dict(case=case)
    if flow == "coo_device":
        I, J, V, n = _coo(case, rng)
        s["ctx"] = L.Context(0)
        s["n"], s["layout"] = n, L.CSC if case["layout"] == "csc" else L.CSR
        s["row"], s["col"], s["val"] = (torch.from_numpy(a).cuda() for a in (I, J, V))
        s["ptr"] = torch.empty(n + 1, dtype=torch.int32, device="cuda")
        s["ind"] = torch.empty(I.size, dtype=torch.int32, device="cuda")
        s["out"] = torch.empty(I.size, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
    elif flow == "coo":
        s["I"], s["J"], s["V"], s["n"] = _coo(case, rng)
        s["ctx"], s["layout"] = L.Context(0), L.CSC if case["layout"] == "csc" else L.CSR
    elif flow == "batch":
        ctx = s["ctx"] = L.Context(0)
        ctx.batch_begin()
        for kind, p, coef in _batch(case, rng):
            f = p["fesp"]
            if kind == "elasticity":
                ctx.batch_add(L.ELAST, L.T6, 3, f.mesh.conn, f.mesh.xy, f.dofnums, f.ndofs(), coef_e=coef, D=p["D"])
            else:
                fe, rule = (L.T3, 1) if kind == "heat_t3" else (L.Q4, 2)
                ctx.batch_add(L.HEAT, fe, rule, f.mesh.conn, f.mesh.xy, f.dofnums, f.ndofs(), coef_e=coef, Q=1.0)
        ctx.batch_build()
    else:
        s["p"] = p = _SETUP[case.get("form", "heat")](case, rng)
        s["am"] = eh.SysmatAssemblerHIP(ctx=L.Context(0))
        s["av"] = eh.SysvecAssemblerHIP(ctx=s["am"].context())
        if "fesp" in p:
            s["n"] = p["fesp"].ndofs()
        else:
            s["n"] = eh.ndofs([p["u"], p["p"]] if "u" in p else [p["ux"], p["uy"], p["p"]])
        if flow == "solve":
            s["nfree"] = p["fesp"].nunknowns()
            s["x0"] = p["fesp"].gathersysvec(np.zeros(s["n"]))
    return s


# ---- one pass ---------------------------------------------------------------------
def _integrate(s, layout):
    c, p, am, av = s["case"], s["p"], s["am"], s["av"]
    eh.start(am, s["n"], s["n"])
    kw = dict(precision=c["precision"], method=c["method"], layout=layout)
    form = c.get("form", "heat")
    if form == "heat":
        eh.start(av, s["n"])
        eh.integrate_heat(am, av, p["fesp"], p["rule"], kappa=p["kappa"], Q=p["Q"], kappa_e=p["kappa_e"], Q_e=p["Q_e"], **kw)
    elif form == "elasticity":
        eh.integrate_elasticity(am, p["fesp"], p["rule"], p["D"], scale_e=p["scale_e"], **kw)
    elif form == "stokes":
        eh.integrate_stokes(am, p["u"], p["p"], p["rule"], mu=p["mu"], **kw)
    else:
        eh.integrate_stokes_reddy(am, p["ux"], p["uy"], p["p"], p["rule"], mu=p["mu"], layout=layout)


def run(s):
    flow = s["case"]["flow"]
    if flow == "coo_device":
        nnz = s["ctx"].sparse_noalloc(s["n"], s["n"], s["val"].numel(), s["row"].data_ptr(), s["col"].data_ptr(),
                                      s["val"].data_ptr(), s["layout"], s["ptr"].data_ptr(), s["ind"].data_ptr(),
                                      s["out"].data_ptr())
        return dict(ptr=s["ptr"], ind=s["ind"][:nnz], val=s["out"][:nnz])
    if flow == "coo":
        s["ctx"].sparse(s["I"], s["J"], s["V"], s["n"], s["n"], s["layout"])
        ptr, ind, val, _, _ = s["ctx"].copy_sparse(base=0)
        return dict(ptr=ptr, ind=ind, val=val)
    if flow == "batch":
        ctx = s["ctx"]
        ctx.batch_assemble()
        return [dict(zip(("ptr", "ind", "val", "F"), ctx.batch_copy(k))) for k in range(s["case"]["problems"])]
    if flow == "solve":
        _integrate(s, "csr")
        F = eh.finish(s["av"])
        x, _, _, _ = s["am"].context().pcg(s["nfree"], F, s["x0"],
                                           precision=L.MIXED if s["case"]["precision"] == "mixed" else L.FP64, tol=1e-10)
        return dict(F=F, x=x)
    _integrate(s, "csc")
    ptr, ind, val, _, _ = s["am"].finish(as_scipy=False)
    out = dict(ptr=ptr, ind=ind, val=val)
    if s["case"]["form"] == "heat":
        out["F"] = eh.finish(s["av"])
    return out


# ---- what a pass cannot do without ----------------------------------------------
def _counts(case):
    """(elements, nodes, element dofs, dofs, entries of the matrix, dofs of the load vector, flops an element)."""
    form, fe, nx, ny, nz = case.get("form", "heat"), case["fe"], case["nx"], case["ny"], case.get("nz", 0)
    cells, nodes = nx * ny, (nx + 1) * (ny + 1)
    edges = nx * (ny + 1) + ny * (nx + 1) + cells  # of the triangles
    if fe == "T4":
        nodes *= nz + 1
        e = nx * ny * nz
        tet_edges = 7 * e + 3 * (nx * ny + ny * nz + nz * nx) + nx + ny + nz
        return 6 * e, nodes, 4, nodes, nodes + 2 * tet_edges, nodes, 400
    if form == "heat":
        e = 2 * cells if fe == "T3" else cells
        nnz = nodes + 2 * (edges + (cells if fe == "Q4" else 0))
        return e, nodes, 3 if fe == "T3" else 4, nodes, nnz, nodes, 90 if fe == "T3" else 700
    if fe == "T6":
        n6 = nodes + edges
        inner, vin = edges - 2 * (nx + ny), (nx - 1) * (ny - 1)  # edges and corners inside
        pairs = 36 * 2 * cells - 9 * inner + vin  # nodes that share an element, by inclusion and exclusion
        if form == "elasticity":
            return 2 * cells, n6, 12, 2 * n6, 4 * pairs, 0, 5000
        return 2 * cells, n6, 15, 2 * n6 + nodes, 4 * pairs + 4 * (18 * 2 * cells - 6 * inner + vin), 0, 6500
    if fe == "T3B":
        return 2 * cells, nodes, 11, 3 * nodes + 4 * cells, 8 * (nodes + 2 * edges) + 2 * cells * 40, 0, 1500
    return cells, nodes, 9, 2 * nodes + cells, 4 * (nodes + 2 * (edges + cells)) + 16 * cells, 0, 1500


def work(case):
    flow = case["flow"]
    if flow in ("coo", "coo_device"):
        nc = 2 if flow == "coo" else 1
        cells, nodes = case["nx"] * case["ny"], (case["nx"] + 1) * (case["ny"] + 1)
        n = 2 * cells * (3 * nc) ** 2
        nnz = (nodes + 2 * (case["nx"] * (case["ny"] + 1) + case["ny"] * (case["nx"] + 1) + cells)) * nc * nc
        wide = 8 if flow == "coo" else 4  # the indices of the result
        return {"bytes": 24.0 * n + (8 + wide) * nnz + wide * nodes * nc, "flops": float(n)}
    if flow == "batch":
        e = case["problems"] * (case["emax"] - case["emin"]) / math.log(case["emax"] / case["emin"])
        return {"bytes": e * (24 + 40 + 16 * 16), "flops": e * 2000.0}
    E, nodes, nd, ndofs, nnz, nf, fl = _counts(case)
    inputs = E * (4.0 * nd + 8) + nodes * 16.0 + ndofs * 4.0
    if flow == "solve":
        its = 3.0 * max(case["nx"], case["ny"]) if case["fe"] == "T3" else 5.0 * max(case["nx"], case["ny"])
        wide = 4 if case["precision"] == "mixed" else 8
        return {"bytes": inputs + nnz * 12.0 + its * ndofs * wide * (nnz / ndofs + 8), "flops": E * float(fl) + its * (2.0 * nnz + 12 * ndofs)}
    return {"bytes": inputs + nnz * 16.0 + ndofs * 8.0 + nf * 8.0, "flops": E * float(fl)}


# ---- the same in 64 bits, by plain torch ---------------------------------------
def _points(fe):
    """Parametric points and weights of the rules above."""
    if fe == "T3":
        return np.array([[1 / 3, 1 / 3]]), np.array([0.5])
    if fe in ("T6", "T3B"):
        return np.array([[2 / 3, 1 / 6], [1 / 6, 2 / 3], [1 / 6, 1 / 6]]), np.full(3, 1 / 6)
    if fe == "T4":
        return np.array([[0.25, 0.25, 0.25]]), np.array([1 / 6])
    a = 0.577350269189626
    return np.array([[i, j] for i in (-a, a) for j in (-a, a)]), np.ones(4)


def _basis(fe, pt):
    """Values and parametric gradients of the basis at one point."""
    if fe == "T4":
        r, s, t = pt
        return np.array([1 - r - s - t, r, s, t]), np.array([[-1, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1.0]])
    r, s = pt
    t = 1 - r - s
    if fe == "T3":
        return np.array([t, r, s]), np.array([[-1, -1], [1, 0], [0, 1.0]])
    if fe == "T3B":
        return np.array([t, r, s, t * r * s]), np.array([[-1, -1], [1, 0], [0, 1.0], [(t - r) * s, (t - s) * r]])
    if fe == "T6":
        dt, dr, ds = np.array([-1.0, -1.0]), np.array([1.0, 0.0]), np.array([0.0, 1.0])
        N = np.array([t * (2 * t - 1), r * (2 * r - 1), s * (2 * s - 1), 4 * r * t, 4 * r * s, 4 * s * t])
        return N, np.array([(4 * t - 1) * dt, (4 * r - 1) * dr, (4 * s - 1) * ds, 4 * (r * dt + t * dr), 4 * (r * ds + s * dr),
                            4 * (s * dt + t * ds)])
    g = np.array([(-1, -1), (1, -1), (1, 1), (-1, 1)])
    return (1 + g[:, 0] * r) * (1 + g[:, 1] * s) / 4, np.stack([g[:, 0] * (1 + g[:, 1] * s), g[:, 1] * (1 + g[:, 0] * r)], 1) / 4


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _quad(fe, mesh, geo):
    """For each point: basis values, spatial gradients (E, basis, dim) and JxW (E)."""
    ng = {"T3": 3, "T6": 6, "Q4": 4, "T4": 4}[geo]
    X = _t(mesh.xy)[_t(mesh.conn[:, :ng]) - 1]
    for pt, w in zip(*_points(fe)):
        N, g = _basis(fe, pt)
        J = torch.einsum("eks,kd->esd", X, _t(_basis(geo, pt)[1]))
        yield _t(N), torch.einsum("kd,eds->eks", _t(g), torch.linalg.inv(J)), torch.linalg.det(J) * w


def _sum_coo(I, J, V, n, csc):
    """The values of the summed matrix in the order of its layout, with its pointers and indices."""
    key = (J * n + I) if csc else (I * n + J)
    key, order = torch.sort(key, stable=True)
    uniq, inv = torch.unique_consecutive(key, return_inverse=True)
    val = torch.zeros(uniq.numel(), dtype=torch.float64, device=V.device).index_add_(0, inv, V[order])
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=V.device)
    ptr[1:] = torch.cumsum(torch.bincount(torch.div(uniq, n, rounding_mode="floor"), minlength=n), 0)
    return ptr, uniq % n, val


def _block_coo(parts, n, csc):
    """parts: (rows (E, a), columns (E, b), blocks (E, a, b))."""
    I = torch.cat([r[:, :, None].expand_as(k).reshape(-1) for r, c, k in parts])
    J = torch.cat([c[:, None, :].expand_as(k).reshape(-1) for r, c, k in parts])
    return _sum_coo(I, J, torch.cat([k.reshape(-1) for _, _, k in parts]), n, csc)


def _exact_heat(p, fe, csc):
    f = p["fesp"]
    E = f.mesh.nelements
    kap = _t(p["kappa_e"]) if p["kappa_e"] is not None else torch.full((E,), p["kappa"], dtype=torch.float64, device="cuda")
    src = _t(p["Q_e"]) if p["Q_e"] is not None else torch.full((E,), p["Q"], dtype=torch.float64, device="cuda")
    ke = fe_ = 0
    for N, g, w in _quad(fe, f.mesh, fe):
        ke = ke + torch.einsum("eis,ejs,e->eij", g, g, w * kap)
        fe_ = fe_ + torch.einsum("i,e->ei", N, w * src)
    d = _t(f.dofnums[:, 0])[_t(f.mesh.conn) - 1] - 1
    F = torch.zeros(f.ndofs(), dtype=torch.float64, device="cuda").index_add_(0, d.reshape(-1), fe_.reshape(-1))
    return _block_coo([(d, d, ke)], f.ndofs(), csc), F


def _vector_dofs(f):
    return (_t(f.dofnums)[_t(f.mesh.conn) - 1] - 1).reshape(f.mesh.nelements, -1)


def _exact_elasticity(p, csc):
    f = p["fesp"]
    ke = _bdb(f.mesh, p["D"])
    d = _vector_dofs(f)
    return _block_coo([(d, d, ke * _t(p["scale_e"])[:, None, None])], f.ndofs(), csc)


def _bdb(mesh, D):
    E, ke = mesh.nelements, 0
    Dt = _t(D)
    for _, g, w in _quad("T6", mesh, "T6"):
        B = torch.zeros(E, 3, 12, dtype=torch.float64, device="cuda")
        B[:, 0, 0::2] = B[:, 2, 1::2] = g[:, :, 0]
        B[:, 1, 1::2] = B[:, 2, 0::2] = g[:, :, 1]
        DB = torch.einsum("ab,ebj->eaj", Dt, B)
        ke = ke + torch.einsum("eai,eaj->eij", B, DB * w[:, None, None])
    return ke


def _exact_stokes(p, csc):
    u, pr = p["u"], p["p"]
    d, dp = _vector_dofs(u), _t(pr.dofnums[:, 0])[_t(pr.mesh.conn) - 1] - 1
    kup = 0
    for (_, g, w), pt in zip(_quad("T6", u.mesh, "T6"), _points("T6")[0]):
        kup = kup - torch.einsum("ei,j,e->eij", g.reshape(g.shape[0], -1), _t(_basis("T3", pt)[0]), w)
    kuu = _bdb(u.mesh, np.diag([2 * p["mu"], 2 * p["mu"], p["mu"]]))
    return _block_coo([(d, d, kuu), (d, dp, kup), (dp, d, kup.transpose(1, 2))], eh.ndofs([u, pr]), csc)


def _exact_reddy(p, fe, csc):
    ux, uy, pr, mu = p["ux"], p["uy"], p["p"], p["mu"]
    dx, dy, dp = (_t(s.element_dofs()) - 1 for s in (ux, uy, pr))
    kxx = kxy = kyy = kxp = kyp = 0
    for (_, g, w), pt in zip(_quad(fe, ux.mesh, "Q4" if fe == "Q4" else "T3"), _points(fe)[0]):
        gx, gy = g[:, :, 0], g[:, :, 1]
        Np = _t(np.ones(1) if fe == "Q4" else _basis("T3", pt)[0])
        xx, yy = torch.einsum("ei,ej,e->eij", gx, gx, mu * w), torch.einsum("ei,ej,e->eij", gy, gy, mu * w)
        kxx, kyy = kxx + 2 * xx + yy, kyy + xx + 2 * yy
        kxy = kxy + torch.einsum("ei,ej,e->eij", gx, gy, mu * w)
        kxp, kyp = kxp - torch.einsum("ei,j,e->eij", gx, Np, w), kyp - torch.einsum("ei,j,e->eij", gy, Np, w)
    tr = lambda k: k.transpose(1, 2)  # noqa: E731
    return _block_coo([(dx, dx, kxx), (dx, dy, kxy), (dy, dx, tr(kxy)), (dy, dy, kyy), (dx, dp, kxp), (dp, dx, tr(kxp)),
                       (dy, dp, kyp), (dp, dy, tr(kyp))], eh.ndofs([ux, uy, pr]), csc)


def _exact_solve(p, fe):
    """Conjugate gradients in 64 bits, three digits beyond the tolerance of the solves."""
    (ptr, ind, val), F = _exact_heat(p, fe, False)
    f = p["fesp"]
    n, nf = f.ndofs(), f.nunknowns()
    x = _t(f.gathersysvec(np.zeros(n)))
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), ptr[1:] - ptr[:-1])
    A = torch.sparse_csr_tensor(ptr, ind, val, size=(n, n))
    free = (torch.arange(n, device="cuda") < nf).double()
    dinv = free / torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, rows[rows == ind], val[rows == ind])
    b = (F - A @ x) * free
    r, z = b.clone(), dinv * b
    q, rz, y = z.clone(), torch.dot(b, dinv * b), torch.zeros_like(b)
    goal = 1e-13 * float(b.norm())
    for it in range(20000):
        w = (A @ q) * free
        a = rz / torch.dot(q, w)
        y += a * q
        r -= a * w
        z = dinv * r
        new = torch.dot(r, z)
        q = z + (new / rz) * q
        rz = new
        if it % 50 == 49 and float(r.norm()) <= goal:
            break
    return dict(F=F, x=x + y)


def exact(case, seed):
    rng = np.random.default_rng([seed, 1])
    flow, csc = case["flow"], case.get("layout", "csc") == "csc"
    if flow in ("coo", "coo_device"):
        I, J, V, n = _coo(case, rng)
        return dict(ptr=None, ind=None, val=_sum_coo(_t(I) - 1, _t(J) - 1, _t(V), n, csc)[2])
    if flow == "batch":
        out = []
        for kind, p, coef in _batch(case, rng):
            if kind == "elasticity":
                out.append(dict(ptr=None, ind=None, val=_exact_elasticity(p, True)[2], F=None))
            else:
                fe = "T3" if kind == "heat_t3" else "Q4"
                m, F = _exact_heat(dict(p, kappa_e=coef, Q_e=None, Q=1.0), fe, True)
                out.append(dict(ptr=None, ind=None, val=m[2], F=F))
        return out
    form = case.get("form", "heat")
    p = _SETUP[form](case, rng)
    if flow == "solve":
        return _exact_solve(p, case["fe"])
    if form == "heat":
        m, F = _exact_heat(p, case["fe"], True)
        return dict(ptr=None, ind=None, val=m[2], F=F)
    m = _exact_elasticity(p, True) if form == "elasticity" else _exact_stokes(p, True) if form == "stokes" else _exact_reddy(p, case["fe"], True)
    return dict(ptr=None, ind=None, val=m[2])
