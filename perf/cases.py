"""The work that is timed: assemblies, solves and training steps through the package's
public entry points, over the sizes, elements, precisions and options it is used with.

A case is a dict of plain values with a "kind":

  operator    AffineFEOperator on a 2-D Q1 mesh, assembled again into the caller's matrix
              and vector (host arrays), then solved: the plain Gridap driver
  new_space   AffineFEOperator from scratch on a scalar Q2 space: pattern, values and
              right-hand side back on the host (first assembly on a new space)
  poisson     3-D Q1 Poisson, assembled and solved by Jacobi-PCG on the device
  fsai        the same with the learned FSAI preconditioner (factor rebuilt each time)
  train       one training step of that preconditioner
  heat        implicit time step: stiffness + mass + Robin boundary + source at the
              quadrature points, solved from the previous solution
  newton      Newton step of the p-Laplacian on an unstructured hexahedral mesh
  tets        P2 on jittered tetrahedra: assembly, then the residual's product A x
  elasticity  vector Q2 elasticity on a Cartesian mesh: assembly, then A x
  mapped      vector Q2 elasticity on a mapped mesh, assembled and solved
  stokes      Taylor-Hood Stokes blocks assembled into the caller's composite matrix

Coefficients, meshes and states are random with the distributions the tests and the
benchmark use.  exact() evaluates the weak forms cell by cell in FP64 torch.
"""
import functools
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gridap.jl_amd"))
import gridap_hip as G  # noqa: E402
from gridap_hip import _lib  # noqa: E402
from gridap_hip import fsai as FS  # noqa: E402
from gridap_hip.boundary import lower_boundary  # noqa: E402

F64, F32 = _lib.GH_PREC_FP64, _lib.GH_PREC_FP32_ELEM
PREC = {"fp64": F64, "fp32": F32}
RTOL = 1e-8  # of the solves: the tolerance the benchmark quotes


def listed():
    return [
        # the reference's own first driver: 64 x 64 quadrilaterals, A and b on the host,
        # then the solve; launches and latency count
        dict(name="operator_2d_64", kind="operator", nx=64, ny=64),
        # a first assembly, everything from the cell tables on: allocation, symbolic phase,
        # values, pattern and values back to the host
        dict(name="new_q2_space_14", kind="new_space", nx=14, ny=13, nz=15),
        # Jacobi-PCG on 64^3 with a smooth random coefficient: the preconditioner baseline
        dict(name="poisson_64", kind="poisson", nx=64, ny=64, nz=64, field="grf"),
        # the headline mesh, 2.1 M cells with an independent coefficient per cell
        dict(name="poisson_128", kind="poisson", nx=128, ny=128, nz=128, field="iid"),
        # the learned preconditioner on the same 64^3 systems, factor rebuilt each time
        dict(name="fsai_64", kind="fsai", nx=64, ny=64, nz=64),
        # its training, one step per instance
        dict(name="train_32", kind="train", nx=32, ny=32, nz=32, probes=4),
        # one implicit step on a ragged box; few iterations, so the assembly counts too
        dict(name="heat_ragged_77", kind="heat", nx=77, ny=64, nz=51, prec="fp64"),
        # nonlinear solve without lattice topology (a mesh generator's numbering)
        dict(name="newton_unstructured_40", kind="newton", nx=40, ny=40, nz=40, p=3.0,
             prec="fp64"),
        # unstructured tetrahedra, FP32 element arithmetic as the benchmark has it
        dict(name="tets_p2_40", kind="tets", nx=40, ny=40, nz=40, prec="fp32"),
        # linear elasticity on the Cartesian lattice, 164 M stored values
        dict(name="elasticity_q2_32", kind="elasticity", nx=32, ny=32, nz=32, prec="fp32"),
        # the same form on a curved mesh (per-point Jacobians), solved
        dict(name="mapped_elasticity_12", kind="mapped", nx=12, ny=11, nz=10, prec="fp64"),
        # a multi-field system, in place
        dict(name="stokes_64", kind="stokes", nx=64, ny=64),
    ]


# sizes per axis a kind is drawn from (log-uniform), and the axes
_RANGE = {"operator": (8, 160, 2), "new_space": (3, 16, 3), "poisson": (8, 100, 3),
          "fsai": (12, 72, 3), "train": (8, 36, 3), "heat": (8, 88, 3), "newton": (6, 44, 3),
          "tets": (4, 40, 3), "elasticity": (4, 30, 3), "mapped": (3, 12, 3),
          "stokes": (8, 72, 2)}


def draw(rng):
    kind = rng.choice(sorted(_RANGE))
    lo, hi, axes = _RANGE[kind]
    base = lo * (hi / lo) ** rng.random()
    # the axes differ by up to a third from each other
    n = [max(2, min(hi, int(round(base * (0.75 + 0.5 * rng.random()))))) for _ in range(axes)]
    case = dict(kind=kind, nx=n[0], ny=n[1])
    if axes == 3:
        case["nz"] = n[2]
    if kind == "poisson":
        case["field"] = rng.choice(["grf", "iid"])
    if kind == "train":
        case["probes"] = rng.choice([1, 2, 4])
    if kind == "newton":
        case["p"] = rng.choice([2.5, 3.0, 4.0])
    if kind in ("heat", "newton", "tets", "elasticity", "mapped"):
        case["prec"] = rng.choice(["fp64", "fp32"])
    return case


def _part(case):
    return tuple(case[k] for k in ("nx", "ny", "nz") if k in case)


# ---- discretisations (host tables: what a program has before it calls the engine) -----


def _warp(x):
    return x + 0.03 * np.prod(np.sin(2 * np.pi * x), axis=-1)[..., None]


_CLAMP = ["tag_01", "tag_03", "tag_05", "tag_07", "tag_13", "tag_15", "tag_17", "tag_19",
          "tag_25"]  # the faces, edges and corners of x = 0


@functools.lru_cache(maxsize=16)
def _disc(kind, part):
    """The mesh, the space's numbering and the tabulation of a kind on a partition."""
    D = len(part)
    d = {"D": D, "part": part, "elem": _lib.GH_REFFE_QK, "ncomp": 1, "xyz": None, "ggrad": None}
    simplex = False
    if kind == "tets":
        model = G.simplexify(G.CartesianDiscreteModel((0, 1) * 3, part)).jittered(7)
        reffe, degree, tags, simplex = G.ReferenceFE(G.lagrangian, G.Float64, 2), 4, "boundary", True
        d["elem"] = _lib.GH_REFFE_PK
    elif kind in ("elasticity", "mapped"):
        model = G.CartesianDiscreteModel((0, 1) * 3, part, map=_warp if kind == "mapped" else None)
        reffe = G.ReferenceFE(G.lagrangian, G.VectorValue[3, G.Float64], 2)
        degree, tags = 4, (_CLAMP if kind == "elasticity" else "boundary")
        d["ncomp"] = 3
    else:
        model = G.CartesianDiscreteModel((0, 1) * D, part)
        reffe, degree, tags = G.ReferenceFE(G.lagrangian, G.Float64, 1), 2, "boundary"
        if kind == "heat":
            tags = []
    V = G.TestFESpace(model, reffe, dirichlet_tags=tags)
    q = G.Quadrature(D, degree, simplex=simplex)
    shp, grad = reffe.tabulate(D, q.coords, simplex=simplex)
    d.update(model=model, order=V.order, qw=q.weights, shp=shp, grad=grad,
             cd=np.asarray(V.cell_dof_ids), nfree=V.nfree, ndiri=V.ndirichlet,
             nloc=V.cell_dof_ids.shape[1], ncells=model.num_cells())
    if kind == "newton":
        # nodes shuffled inside runs of 64 ids: no lattice topology, generator-like locality
        nn = model.num_nodes()
        rng = np.random.default_rng(13)
        perm = np.arange(nn)
        for k in range(0, nn, 64):
            perm[k:k + 64] = k + rng.permutation(min(64, nn - k))
        xyz = np.empty((nn, D))
        xyz[perm] = _warp(model.node_coordinates())
        cn = perm[model.cell_node_ids() - 1] + 1
        isd = np.zeros(nn, dtype=bool)
        isd[perm] = V.node_and_comp_to_dof[:, 0] < 0
        ids = np.empty(nn, dtype=np.int64)
        ids[~isd] = np.arange(1, np.count_nonzero(~isd) + 1)
        ids[isd] = -np.arange(1, np.count_nonzero(isd) + 1)
        d.update(xyz=xyz, cn=cn.astype(np.int32), cd=ids[cn - 1].astype(np.int32))
    elif kind in ("tets", "mapped"):
        d.update(xyz=model.node_coordinates(), cn=model.cell_node_ids())
    # gradients of the geometry map's basis at the points
    d["ggrad"] = G.ReferenceFE(G.lagrangian, G.Float64, 1).tabulate(D, q.coords,
                                                                   simplex=simplex)[1]
    if kind == "heat":
        trian = G.BoundaryTriangulation(model, model.get_face_labeling(), tags="boundary")
        v, u = G.get_fe_basis(V), G.get_trial_fe_basis(G.TrialFESpace(V))
        dG = G.Measure(trian, 2)
        fac = lower_boundary(model, reffe, G.integrate(1.0 * v * u, dG).terms,
                             G.integrate(1.0 * v, dG).terms)["faces"]
        d["faces"] = fac
        d["fx"] = fac.x
    return d


def _ptrs(table):
    return (np.arange(table.shape[0] + 1, dtype=np.int64) * table.shape[1] + 1).astype(np.int32)


def _context(d):
    ctx = _lib.Context(0)
    if d["xyz"] is None:
        ctx.mesh_cartesian(d["model"].origin, d["model"].sizes, d["part"])
    else:
        ctx.mesh_upload(d["xyz"], d["cn"].ravel(), _ptrs(d["cn"]))
    ctx.space_upload(d["elem"], d["order"], d["ncomp"], d["cd"].ravel(), _ptrs(d["cd"]),
                     d["nfree"], d["ndiri"])
    ctx.reffe_tabulation(d["qw"], d["shp"], d["grad"])
    if d["xyz"] is not None and d["elem"] == _lib.GH_REFFE_QK and d["order"] == 2:
        ctx.geometry_tabulation(d["ggrad"])
    ctx.symbolic()
    return ctx


# ---- inputs ----------------------------------------------------------------------------


def _grf(seed, part, sizes):
    """exp of a smooth Gaussian random field at the cell centres (random Fourier modes)."""
    omega, phase, amp = FS.grf_modes(seed)
    ax = [(np.arange(n) + 0.5) * h for n, h in zip(part, sizes)]
    # cos(w.x + p) summed over modes, separable phases: one small product per axis
    e = [np.exp(1j * np.outer(omega[:, k], a)) for k, a in enumerate(ax)]
    g = np.einsum("mx,my,mz->zyx", e[0] * np.exp(1j * phase)[:, None], e[1], e[2],
                  optimize=True).real
    return np.exp(amp * g).ravel()


def _inputs(case, seed):
    """The random data of a case, from the seed alone."""
    kind, part = case["kind"], _part(case)
    rng = np.random.default_rng([1000003, int(seed)])
    nc = int(np.prod(part))
    if kind in ("operator", "new_space"):
        return dict(kappa=np.exp(rng.standard_normal(nc)), f=rng.uniform(-1, 1, nc))
    if kind == "stokes":
        c = rng.uniform(0.5, 2.0, 3)
        return dict(coef=c)
    d = _disc(kind, part)
    C, N = d["ncells"], d["nfree"]
    if kind == "poisson":
        k = _grf(seed, part, d["model"].sizes) if case["field"] == "grf" else \
            np.exp(rng.standard_normal(C))
        return dict(kappa=k, f=1.0 + 0.5 * rng.uniform(-1, 1, C))
    if kind in ("fsai", "train"):
        return dict(kappa=_grf(seed, part, d["model"].sizes))
    if kind == "heat":
        nq = len(d["qw"])
        fx = d["fx"]
        return dict(kappa=np.exp(0.5 * rng.standard_normal(C)),
                    sigma=np.full(C, 0.25 * float(np.mean(part)) ** 2) * rng.uniform(0.5, 2, C),
                    fq=rng.uniform(-1, 1, (C, nq)), alpha=rng.uniform(1, 3, fx.shape[0]),
                    g=np.sin(3 * fx[..., 0]) + fx[..., 1] * rng.uniform(0.5, 2),
                    u0=rng.uniform(-1, 1, N))
    if kind == "newton":
        # a state with an O(1) gradient everywhere, as an iterate has
        x = d["xyz"]
        c = rng.uniform(0.5, 1.5, 3)
        nodal = 0.7 * x @ c + 0.1 * np.sin(4 * x[:, 0] * c[0]) * np.cos(3 * x[:, 1])
        u, ud = np.zeros(N), np.zeros(d["ndiri"])
        dof, val = d["cd"].ravel().astype(np.int64), nodal[d["cn"].ravel() - 1]
        u[dof[dof > 0] - 1] = val[dof > 0]
        ud[-dof[dof < 0] - 1] = val[dof < 0]
        return dict(kappa=np.exp(0.3 * rng.standard_normal(C)), f=rng.uniform(-1, 1, C), u=u, ud=ud)
    if kind == "tets":
        return dict(kappa=np.exp(rng.standard_normal(C)), f=rng.uniform(-1, 1, C),
                    ud=rng.uniform(-1, 1, d["ndiri"]), x=rng.standard_normal(N))
    if kind == "elasticity":
        return dict(kappa=np.exp(0.5 * rng.standard_normal(C)), x=rng.standard_normal(N))
    return dict(kappa=np.exp(0.5 * rng.standard_normal(C)))  # mapped


_BODY = (0.0, 0.0, -1.0)
_NU = 0.3
_TRAIN_LR = 2e-3


def _q2_space(part):
    model = G.CartesianDiscreteModel((0, 1) * 3, part)
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 2), dirichlet_tags="boundary")
    return model, V


_new_space = functools.lru_cache(maxsize=8)(_q2_space)


@functools.lru_cache(maxsize=8)
def _stokes_spaces(part):
    model = G.CartesianDiscreteModel((0, 2, 0, 2), part)
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.VectorValue[2, G.Float64], 2),
                      dirichlet_tags="boundary")
    Q = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1), dirichlet_tags="tag_1")
    return model, V, Q


def _diri_2d(x):
    return x[..., 0] + 2 * x[..., 1]


def _stokes_u(x):
    return np.stack([x[..., 0] ** 2 + 2 * x[..., 1] ** 2, -x[..., 0] ** 2], axis=-1)


def _stokes_p(x):
    return x[..., 0] + 3 * x[..., 1]


def prepare(case, seed):
    kind, part = case["kind"], _part(case)
    z = _inputs(case, seed)
    s = {"kind": kind}
    if kind in ("operator", "new_space"):
        if kind == "operator":
            model = G.CartesianDiscreteModel((0, 1) * 2, part)
            V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1),
                              dirichlet_tags="boundary")
            U, degree = G.TrialFESpace(V, _diri_2d), 2
        else:
            model, V = _new_space(part)
            U, degree = G.TrialFESpace(V), 4
        omega = G.Triangulation(model)
        dx = G.Measure(omega, degree)
        k, f = G.CellField(z["kappa"], omega), G.CellField(z["f"], omega)
        s.update(U=U, V=V, a=lambda u, v: G.integrate(k * G.inner(G.gradient(v), G.gradient(u)), dx),
                 l=lambda v: G.integrate(f * v, dx))
        if kind == "operator":
            s["assem"] = G.SparseMatrixAssembler(U, V)
            s["A"], s["b"] = G.assemble_matrix_and_vector(s["a"], s["l"], U, V, s["assem"])
            s["solver"] = G.PCGSolver(rtol=1e-10)
        return s
    if kind == "stokes":
        model, V, Q = _stokes_spaces(part)
        U, P = G.TrialFESpace(V, _stokes_u), G.TrialFESpace(Q, _stokes_p)
        X, Y = G.MultiFieldFESpace([U, P]), G.MultiFieldFESpace([V, Q])
        dx = G.Measure(G.Triangulation(model), 2)
        mu, f0, f1 = (float(c) for c in z["coef"])
        s["a"] = lambda u, v: G.integrate(mu * G.inner(G.gradient(v[0]), G.gradient(u[0])) -
                                          G.divergence(v[0]) * u[1] + v[1] * G.divergence(u[0]), dx)
        s["l"] = lambda v: G.integrate(G.dot(v[0], G.VectorValue(-f0, f1)) +
                                       v[1] * (lambda x: 2.0 * x[..., 0]), dx)
        s["assem"] = G.SparseMatrixAssembler(X, Y)
        # the second assembly composes on the device: a program in a loop is past it
        s["A"], s["b"] = G.assemble_matrix_and_vector(s["a"], s["l"], X, Y, s["assem"])
        G.assemble_matrix_and_vector_inplace(s["a"], s["l"], s["A"], s["b"], s["assem"])
        return s
    d = _disc(kind, part)
    ctx = s["ctx"] = _context(d)
    s["prec"] = PREC[case.get("prec", "fp64")]
    if kind in ("poisson", "fsai", "train"):
        ctx.coef_upload(z["kappa"], z.get("f"), None)
        if kind != "poisson":
            FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).attach(ctx)
        if kind == "train":
            s.update(probes=case["probes"], step=0, seed=int(seed))
            ctx.assemble(_lib.GH_FORM_DIFFUSION, F64)
    elif kind == "heat":
        fac = d["faces"]
        ctx.coef_upload(z["kappa"], None, None)
        ctx.mass_upload(z["sigma"])
        ctx.source_qp_upload(z["fq"])
        ctx.face_tabulation(fac.qw, fac.shp, fac.grad)
        ctx.boundary_upload(fac.cells + 1, fac.sides + 1, z["alpha"], None, z["g"], None)
        s["u0"] = z["u0"]
    elif kind == "newton":
        ctx.coef_upload(z["kappa"], z["f"], None)
        ctx.plaplacian_params(case["p"])
        s.update(u=z["u"], ud=z["ud"])
    elif kind == "tets":
        ctx.coef_upload(z["kappa"], z["f"], z["ud"])
        s["x"] = z["x"]
    else:
        ctx.coef_upload(z["kappa"], None, None)
        ctx.elasticity_params(_NU, _BODY)
        s["x"] = z.get("x")
    return s


def run(s):
    kind = s["kind"]
    if kind == "operator":
        A, b = G.assemble_matrix_and_vector_inplace(s["a"], s["l"], s["A"], s["b"], s["assem"])
        return {"nzval": A.nzval, "b": b, "x": s["solver"].solve(s["assem"], b, A)}
    if kind == "new_space":
        op = G.AffineFEOperator(s["a"], s["l"], s["U"], s["V"])
        A = op.get_matrix()
        return {"colptr": A.colptr, "rowval": A.rowval, "nzval": A.nzval, "b": op.get_vector()}
    if kind == "stokes":
        A, b = G.assemble_matrix_and_vector_inplace(s["a"], s["l"], s["A"], s["b"], s["assem"])
        return {"nzval": A.nzval, "b": b}
    ctx = s["ctx"]
    if kind == "poisson":
        ctx.assemble(_lib.GH_FORM_DIFFUSION, s["prec"])
        return {"x": ctx.pcg(rtol=RTOL)[0]}
    if kind == "fsai":
        ctx.assemble(_lib.GH_FORM_DIFFUSION, s["prec"])
        ctx.fsai_build()
        return {"x": ctx.pcg(rtol=RTOL, precond=_lib.GH_PRECOND_FSAI)[0]}
    if kind == "train":
        s["step"] += 1
        loss = ctx.fsai_train_step(s["probes"], 1000003 * s["step"] + s["seed"], _TRAIN_LR)
        return {"loss": loss, "weights": ctx.mlp_get()}
    if kind == "heat":
        ctx.assemble(_lib.GH_FORM_DIFFUSION, s["prec"])
        return {"x": ctx.pcg(x0=s["u0"], rtol=RTOL)[0]}
    if kind == "newton":
        ctx.fefunction_upload(s["u"], s["ud"])
        ctx.assemble(_lib.GH_FORM_PLAPLACIAN, s["prec"])
        _, r = ctx.values_get(want_nz=False)
        return {"residual": r, "dx": ctx.pcg(b=-r, rtol=RTOL)[0]}
    if kind == "tets":
        ctx.assemble(_lib.GH_FORM_DIFFUSION, s["prec"])
    else:
        ctx.assemble(_lib.GH_FORM_ELASTICITY, s["prec"])
        if kind == "mapped":
            return {"x": ctx.pcg(rtol=RTOL)[0]}
    _, b = ctx.values_get(want_nz=False)
    return {"b": b, "Ax": ctx.spmv(s["x"])}


# ---- minimal work ----------------------------------------------------------------------


def _sizes(case):
    """(cells, unknowns, stored values, nodes per cell) of a case, to within the boundary."""
    kind, n = case["kind"], _part(case)
    C = int(np.prod(n))
    p = lambda k, c: int(np.prod([k * m + c for m in n]))
    if kind in ("operator", "poisson", "fsai", "train", "newton"):
        return C, p(1, -1), p(3, -5), 2 ** len(n)
    if kind == "heat":
        return C, p(1, 1), p(3, 1), 8
    if kind == "new_space":
        return C, p(2, -1), p(8, -7), 27
    if kind == "tets":
        return 6 * C, p(2, -1), 230 * C, 10
    if kind == "stokes":
        return C, 2 * p(2, -1) + p(1, 1), 4 * p(8, -7) + 2 * 2 * p(5, 1), 22
    return C, 3 * p(2, 0), 9 * p(8, 0), 81


def _iterations(case):
    """CG iterations to the tolerance, about what these systems take."""
    n = float(np.mean(_part(case)))
    return {"operator": 3.6 * n, "poisson": (3.0 if case.get("field") == "grf" else 2.6) * n,
            "fsai": 1.8 * n, "heat": 25.0, "newton": 3.0 * n, "mapped": 60 + 9.0 * n
            }.get(case["kind"], 0)


def work(case):
    kind = case["kind"]
    C, N, nnz, nl = _sizes(case)
    if kind == "train":
        w = 10 * 64 + 64 * 64 * 2 + 64 * 36
        # forward, input and weight gradients of the network per cell; per probe two products
        # with A and four with the factor's half
        return {"bytes": 8 * nnz + 8 * C + 4 * 4 * 11364 + 24 * N * case["probes"],
                "flops": 6 * C * w + case["probes"] * nnz * 10}
    it = _iterations(case)
    # the assembly writes A and b once from one coefficient per cell; an iteration reads A's
    # values and p, x, r, z and writes p, x, r, z; the factor has half of A's entries in FP32
    per = 8 * nnz + 8 * 8 * N + (4 * nnz if kind == "fsai" else 0)
    b = 8 * nnz + 8 * N + 16 * C + 4 * nl * C + it * per
    f = 2 * nl * nl * C + it * (2 * nnz + 12 * N + (2 * nnz if kind == "fsai" else 0))
    if kind in ("tets", "elasticity"):
        b += 8 * nnz + 16 * N   # A x
        f += 2 * nnz
    if kind == "new_space":
        b += 8 * nnz + 8 * N    # the pattern
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """About four times what run() shows against exact() over the ranges of draw()."""
    kind, fp32 = case["kind"], case.get("prec") == "fp32"
    if kind in ("operator", "poisson", "fsai"):
        # iterates stopped at a relative residual of 1e-8 (operator: 1e-10, larger
        # systems): another stopping iteration is within this
        return {"rel": 1e-8, "max": 4e-8}
    if kind in ("heat", "newton", "mapped"):
        return {"rel": 7e-7, "max": 2.5e-6} if fp32 else {"rel": 5e-8, "max": 2e-7}
    if kind == "train":
        return {"rel": 2e-6, "max": 2e-4}  # FP32 network, gradient and optimiser
    if fp32:
        return {"rel": 4e-7, "max": 2e-6}
    return {"rel": 1e-14, "max": 2e-13}


# ---- FP64 evaluation, cell by cell --------------------------------------------------------


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev(), dtype=dtype)


def _geometry(d, cells=None):
    """w |det J| [c, q] and physical gradients [c, q, a, D] of the cells."""
    grad, qw = _t(d["grad"]), _t(d["qw"])
    if d["xyz"] is None:
        h = _t(d["model"].sizes)
        g = grad / h
        return (qw * h.prod())[None], g[None]
    cn = torch.as_tensor(d["cn"].astype(np.int64) - 1, device=_dev())
    if cells is not None:
        cn = cn[cells]
    X = _t(d["xyz"])[cn]                                          # c, v, D
    J = torch.einsum("cvi,qvj->cqij", X, _t(d["ggrad"]))          # dx_i / dxi_j
    Ji = torch.linalg.inv(J)
    g = torch.einsum("cqji,qaj->cqai", Ji, grad)
    return torch.linalg.det(J).abs() * qw, g


def _blocks(C, per, limit=64_000_000):
    step = max(1, min(C, limit // per))
    return [slice(i, min(C, i + step)) for i in range(0, C, step)]


def _cells(d, w, g, k, sigma=None, elastic=False, body=None, src=None, state=None, p=None):
    """Element matrices and loads of a run of cells with weights w and gradients g."""
    shp, D, n, nn = _t(d["shp"]), d["D"], k.shape[0], d["shp"].shape[1]
    w, g = w.expand(n, -1), g.expand(n, -1, -1, -1)
    if elastic:
        P = torch.einsum("cq,cqai,cqbj->cijab", w, g, g)
        lam, mu = _NU / ((1 + _NU) * (1 - 2 * _NU)), 1 / (2 * (1 + _NU))
        tr = P.diagonal(dim1=1, dim2=2).sum(-1)
        B = lam * P + mu * P.transpose(1, 2)
        for i in range(D):
            B[:, i, i] += mu * tr
        K = k[:, None, None] * B.permute(0, 1, 3, 2, 4).reshape(n, nn * D, nn * D)
        return K, torch.cat([body[i] * (w @ shp) for i in range(D)], dim=1)
    if state is not None:
        gu = torch.einsum("cqad,ca->cqd", g, state)
        a = gu.norm(dim=-1)
        ga = torch.einsum("cqad,cqd->cqa", g, gu)
        wk = w * k[:, None]
        K = (torch.einsum("cq,cqad,cqbd->cab", wk * a ** (p - 2), g, g) +
             torch.einsum("cq,cqa,cqb->cab", wk * (p - 2) * a ** (p - 4), ga, ga))
        return K, torch.einsum("cq,cqa->ca", wk * a ** (p - 2), ga) - (w * src) @ shp
    K = k[:, None, None] * torch.einsum("cq,cqad,cqbd->cab", w, g, g)
    if sigma is not None:
        K += sigma[:, None, None] * torch.einsum("cq,qa,qb->cab", w, shp, shp)
    return K, (w * src) @ shp


def _elements(d, kappa, sigma=None, elastic=False, body=None, src=None, state=None, p=None):
    """Element matrices [c, nloc, nloc] and loads [c, nloc] of all cells."""
    C, nq, nn = d["ncells"], len(d["qw"]), d["shp"].shape[1]
    if d["xyz"] is None:
        # every cell has the Jacobian diag(h): one reference matrix, scaled
        w, g = _geometry(d)
        one = torch.ones(1, dtype=torch.float64, device=_dev())
        shp = _t(d["shp"])
        K, F = _cells(d, w, g, one, None, elastic, body, one[:, None])
        K = kappa[:, None, None] * K
        if sigma is not None:
            K += sigma[:, None, None] * torch.einsum("q,qa,qb->ab", w[0], shp, shp)
        return K, F.expand(C, -1) if elastic else (src * w) @ shp
    Ks, Fs = [], []
    cut = lambda v, s: v if v is None or v.shape[0] == 1 else v[s]
    for s in _blocks(C, nq * nn * d["D"] + 3 * (nn * d["ncomp"]) ** 2):
        K, F = _cells(d, *_geometry(d, s), kappa[s], cut(sigma, s), elastic, body, cut(src, s),
                      cut(state, s), p)
        Ks.append(K)
        Fs.append(F)
    return torch.cat(Ks), torch.cat(Fs)


def _mul(K, x):
    """K x of every cell."""
    return (K * x[:, None, :]).sum(-1)


class _System:
    """The assembled operator as a sum over cells."""

    def __init__(self, d, K, F=None, ud=None):
        cd = torch.as_tensor(d["cd"].astype(np.int64), device=_dev())
        self.n, self.K = d["nfree"], K
        self.free = cd > 0
        self.at = torch.where(self.free, cd - 1, torch.full_like(cd, self.n))
        # the cell entries of every dof, padded with one past the last entry
        at = self.at.reshape(-1)
        order = torch.argsort(at, stable=True)
        first = torch.searchsorted(at[order], torch.arange(self.n + 1, device=at.device))
        k = int(first[-1])
        rank = torch.arange(k, device=at.device) - first[at[order[:k]]]
        self.entries = torch.full((self.n, int(rank.max()) + 1), at.numel(), device=at.device)
        self.entries[at[order[:k]], rank] = order[:k]
        if F is not None:
            if ud is not None:
                loc = torch.where(cd < 0, ud[(-cd - 1).clamp_min(0)], torch.zeros_like(F))
                F = F - _mul(K, loc)
            self.b = self.sum(F)

    def sum(self, v):
        v = v.reshape(-1)
        return torch.cat([v, v.new_zeros(1)])[self.entries].sum(1)

    def local(self, x):
        return torch.cat([x, x.new_zeros(1)])[self.at]

    def apply(self, x):
        return self.sum(_mul(self.K, self.local(x)))

    def diagonal(self):
        return self.sum(self.K.diagonal(dim1=1, dim2=2))

    def solve(self, b, x=None, tol=1e-12):
        """Jacobi-CG far below the tolerance of the case."""
        x = torch.zeros_like(b) if x is None else x.clone()
        d = 1 / self.diagonal()
        r = b - self.apply(x)
        z = d * r
        p, rz, stop = z.clone(), float(r @ z), tol * float(b.norm())
        for it in range(4000):
            q = self.apply(p)
            a = rz / float(p @ q)
            x += a * p
            r -= a * q
            if it % 10 == 0 and float(r.norm()) <= stop:
                break
            z = d * r
            rz, old = float(r @ z), rz
            p = z + (rz / old) * p
        return x


def _csc(nrows, rows, cols, vals, ncols):
    """colptr, rowval (1-based) and nzval of summed triplets, duplicates in any order."""
    key, inv = torch.unique(cols * nrows + rows, return_inverse=True)
    nz = torch.zeros(key.numel(), dtype=torch.float64, device=vals.device)
    nz.index_add_(0, inv, vals)
    cnt = torch.bincount(key // nrows, minlength=ncols)
    cp = torch.cat([cnt.new_ones(1), 1 + torch.cumsum(cnt, 0)])
    return cp, key % nrows + 1, nz


def _triplets(cr, cc, K):
    """Free (row, column, value) of element matrices K [c, nr, nc]."""
    r = cr[:, :, None].expand(K.shape)
    c = cc[:, None, :].expand(K.shape)
    ok = (r > 0) & (c > 0)
    return r[ok] - 1, c[ok] - 1, K[ok]


def _scalar_disc(model, V, degree):
    q = G.Quadrature(model.D, degree)
    shp, grad = V.reffe.tabulate(model.D, q.coords)
    return dict(D=model.D, ncomp=V.ncomp, model=model, xyz=None, qw=q.weights, shp=shp, grad=grad,
                cd=np.asarray(V.cell_dof_ids), nfree=V.nfree, ndiri=V.ndirichlet,
                ncells=model.num_cells())


def _exact_train(case, seed, d, z, system):
    """Loss and weights after one step, by automatic differentiation in FP64."""
    C, n = d["ncells"], d["nfree"]
    w0 = FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).params.astype(np.float32)
    w = _t(torch.as_tensor(w0).to(torch.bfloat16).double().numpy()).requires_grad_(True)
    cut, at = [], 0
    for shape in ((64, 10), (64,), (64, 64), (64,), (64, 64), (64,), (36, 64), (36,)):
        m = int(np.prod(shape))
        cut.append(w[at:at + m].reshape(shape))
        at += m
    dg = system.diagonal()
    diag = torch.cat([dg, dg.new_full((1,), float("inf"))])[system.at]
    kaa = system.K.diagonal(dim1=1, dim2=2)
    logh = float(np.log(np.prod(d["model"].sizes)) / 3)
    h = torch.cat([kaa / diag, _t(z["kappa"]).log()[:, None],
                   torch.full((C, 1), logh, dtype=torch.float64, device=_dev())], 1)
    for i in range(0, 6, 2):
        h = torch.nn.functional.gelu(h @ cut[i].T + cut[i + 1])
    y = h @ cut[6].T + cut[7]
    L = torch.zeros(C, 8, 8, dtype=torch.float64, device=_dev())
    ia = [(a, b) for a in range(8) for b in range(a)]
    L[:, [a for a, _ in ia], [b for _, b in ia]] = y[:, 8:]
    dexp = system.sum(y[:, :8]).exp()
    s = dg ** -0.5

    def gmul(v):
        v = s * v
        return dexp * v + system.sum(_mul(L, system.local(v)))

    def gt(v):
        return s * (dexp * v +
                    system.sum(_mul(L.transpose(1, 2), system.local(v))))

    def mix(x):
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))

    m, loss = case["probes"], 0.0
    i = np.arange(1, n + 1, dtype=np.uint64)
    for k in range(m):
        t = np.uint64(1000003 + int(seed)) + np.uint64(0x9E3779B97F4A7C15) * (
            np.uint64(k) * np.uint64(0x100000001) + i)
        v = _t(np.where(mix(t) & np.uint64(1), 1.0, -1.0))
        r = v - gmul(system.apply(gt(v)))
        loss = loss + r @ r
    loss = loss / (m * n)
    (g,) = torch.autograd.grad(loss, w)
    new = _t(w0) - _TRAIN_LR * g / (g.abs() + 1e-8)
    return {"loss": float(loss.detach()), "weights": new.detach()}


def exact(case, seed):
    kind, part = case["kind"], _part(case)
    z = _inputs(case, seed)
    if kind == "operator":
        model = G.CartesianDiscreteModel((0, 1) * 2, part)
        V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1),
                          dirichlet_tags="boundary")
        d = _scalar_disc(model, V, 2)
        ud = _t(G.TrialFESpace(V, _diri_2d).dirichlet_values())
    elif kind == "new_space":
        model, V = _new_space(part)
        d, ud = _scalar_disc(model, V, 4), None
    if kind in ("operator", "new_space"):
        K, F = _elements(d, _t(z["kappa"]), src=_t(z["f"])[:, None])
        S = _System(d, K, F, ud)
        cd = _t(d["cd"], torch.int64)
        cp, rv, nz = _csc(S.n, *_triplets(cd, cd, K), S.n)
        if kind == "operator":
            return {"nzval": nz, "b": S.b, "x": S.solve(S.b)}
        return {"colptr": cp, "rowval": rv, "nzval": nz, "b": S.b}
    if kind == "stokes":
        return _exact_stokes(part, z)
    d = _disc(kind, part)
    kap = _t(z["kappa"])
    if kind in ("poisson", "fsai", "train"):
        K, F = _elements(d, kap, src=_t(z.get("f", np.ones(d["ncells"])))[:, None])
        S = _System(d, K, F)
        if kind == "train":
            return _exact_train(case, seed, d, z, S)
        return {"x": S.solve(S.b)}
    if kind == "heat":
        K, F = _elements(d, kap, sigma=_t(z["sigma"]), src=_t(z["fq"]))
        fac = d["faces"]
        h = np.asarray(d["model"].sizes)
        area = np.prod(h) / h[fac.axis]
        w = _t(area)[:, None] * _t(fac.qw) * _t(z["alpha"])[:, None]
        ph = _t(fac.shp[fac.sides])
        c = torch.as_tensor(fac.cells, device=_dev())
        K.index_add_(0, c, torch.einsum("fq,fqa,fqb->fab", w, ph, ph))
        F.index_add_(0, c, torch.einsum("fq,fqa->fa", _t(area)[:, None] * _t(fac.qw) * _t(z["g"]),
                                        ph))
        S = _System(d, K, F)
        return {"x": S.solve(S.b, _t(z["u0"]))}
    if kind == "newton":
        S = _System(d, None)
        u = torch.cat([_t(z["u"]), _t(z["ud"])])
        cd = _t(d["cd"], torch.int64)
        uc = u[torch.where(cd > 0, cd - 1, d["nfree"] - cd - 1)]
        K, F = _elements(d, kap, src=_t(z["f"])[:, None], state=uc, p=case["p"])
        S.K = K
        r = S.sum(F)
        return {"residual": r, "dx": S.solve(-r)}
    if kind == "tets":
        K, F = _elements(d, kap, src=_t(z["f"])[:, None])
        S = _System(d, K, F, _t(z["ud"]))
    else:
        K, F = _elements(d, kap, elastic=True, body=_BODY)
        S = _System(d, K, F)
        if kind == "mapped":
            return {"x": S.solve(S.b)}
    return {"b": S.b, "Ax": S.apply(_t(z["x"]))}


def _exact_stokes(part, z):
    model, V, Q = _stokes_spaces(part)
    mu, f0, f1 = (float(c) for c in z["coef"])
    # vector Q2: the scalar element matrix on each component
    d = _scalar_disc(model, V, 2)
    w, g = _geometry(d)
    nn, C = 9, d["ncells"]
    Ks = mu * torch.einsum("cq,cqad,cqbd->cab", w, g, g)[0]
    K = torch.zeros(18, 18, dtype=torch.float64, device=_dev())
    K[:9, :9] = K[9:, 9:] = Ks
    q1 = _t(Q.reffe.tabulate(2, G.Quadrature(2, 2).coords)[0])
    B = torch.cat([torch.einsum("q,qp,qa->pa", w[0], q1, g[0, :, :, i]) for i in range(2)], 1)
    vd, pd = _t(V.cell_dof_ids, torch.int64), _t(Q.cell_dof_ids, torch.int64)
    nv, npr = V.nfree, Q.nfree
    shift = lambda c: torch.where(c > 0, c + nv, c)
    n = nv + npr
    tr = [_triplets(vd, vd, K.expand(C, -1, -1)),
          _triplets(shift(pd), vd, B.expand(C, -1, -1)),
          _triplets(vd, shift(pd), -B.T.expand(C, -1, -1))]
    _, _, nz = _csc(n, *(torch.cat([t[k] for t in tr]) for k in range(3)), n)
    shp = _t(d["shp"])
    m = torch.einsum("q,qa->a", w[0], shp)
    Fv = torch.cat([-f0 * m, f1 * m]).expand(C, -1).clone()
    qx = _t(G.Quadrature(2, 2).coords)
    cx = _t(np.arange(C) % part[0])
    x0 = (cx[:, None] + qx[:, 0]) * float(model.sizes[0])
    Fp = torch.einsum("cq,qp->cp", w * 2.0 * x0, q1)
    ud = _t(G.TrialFESpace(V, _stokes_u).dirichlet_values())
    qd = _t(G.TrialFESpace(Q, _stokes_p).dirichlet_values())
    uc = torch.where(vd < 0, ud[(-vd - 1).clamp_min(0)], ud.new_zeros(1))
    pc = torch.where(pd < 0, qd[(-pd - 1).clamp_min(0)], qd.new_zeros(1))
    Fv = Fv - uc @ K.T + pc @ B
    Fp = Fp - uc @ B.T
    b = torch.zeros(n + 1, dtype=torch.float64, device=_dev())
    for cd, F in ((vd, Fv), (shift(pd), Fp)):
        b.index_add_(0, torch.where(cd > 0, cd - 1, n).reshape(-1), F.reshape(-1))
    return {"nzval": nz, "b": b[:-1]}
