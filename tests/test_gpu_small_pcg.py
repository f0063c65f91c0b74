"""The one-workgroup solve of small systems against the general kernels on the same
system: sizes at the edges of its row counts (512, 1024, 2048, 4096), rows inside and past
the entries held in registers, sizes past its rule, an uneven matrix that it declines,
restarts, iteration limits and a solve taken up by a second launch (needs an MI355X).

Both run the same recurrences in FP64 and differ in the grouping of the dot products:
the iteration counts agree to one and the solutions, stopped at 1e-10, to 1e-10 times the
condition number (below 1e4 here)."""
import os

import numpy as np
import pytest

import gridap_hip as G
from gridap_hip import _lib

pytestmark = pytest.mark.gpu


class env:
    def __init__(self, **kw):
        self.kw = kw

    def __enter__(self):
        self.old = {k: os.environ.get(k) for k in self.kw}
        os.environ.update(self.kw)

    def __exit__(self, *a):
        for k, v in self.old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


def small(ctx, **kw):
    r = ctx.pcg(**kw)
    assert ctx.solve_form() == _lib.GH_SOLVE_WORKGROUP
    return r


def general(ctx, **kw):
    with env(GRIDAP_HIP_SMALL_PCG="0", GRIDAP_HIP_RESIDENT_PCG="0"):
        r = ctx.pcg(**kw)
    assert ctx.solve_form() in (_lib.GH_SOLVE_ROWS, _lib.GH_SOLVE_STENCIL)
    return r


def system(D, part, order=1, ncomp=1, tags="boundary", seed=0, spread=0.5):
    model = G.CartesianDiscreteModel((0, 1) * D, part)
    T = G.VectorValue[D, G.Float64] if ncomp > 1 else G.Float64
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, T, order), dirichlet_tags=tags)
    U = G.TrialFESpace(V)
    Ω = G.Triangulation(model)
    dx = G.Measure(Ω, 2 * order)
    k = G.CellField(np.exp(np.random.default_rng(seed).normal(0, spread, model.num_cells())), Ω)
    if ncomp > 1:
        s = G.IsotropicStress(k, 0.3)
        a = lambda u, v: G.integrate(G.inner(G.ε(v), s(G.ε(u))), dx)
    else:
        a = lambda u, v: G.integrate(k * G.inner(G.gradient(v), G.gradient(u)), dx)
    assem = G.SparseMatrixAssembler(U, V)
    return G.assemble_matrix(a, assem, U, V), assem.ctx, assem


# 2-D Q1 rows of 9, 3-D Q1 of 27 (past the registers' 18 from 1025 rows), scalar Q2 (to 125;
# 2209 rows of up to 25, past the nine kept there), vector Q2; 1, 2, 512, 528, 1024, 1056, 2048, 2070, 4032, 4096 rows and past the rule
CASES = [(2, (2, 2)), (2, (3, 2)), (2, (33, 17)), (2, (34, 17)), (2, (33, 33)), (2, (33, 34)),
         (2, (65, 33)), (2, (47, 46)), (2, (65, 64)), (2, (65, 65)), (2, (66, 65)),
         (3, (11, 11, 11)), (3, (9, 14, 13)), (3, (16, 16, 16)), (3, (4, 4, 4), 2), (2, (24, 24), 2),
         (3, (2, 2, 2), 2, 3, ["tag_25"]), (2, (9, 8), 2, 2)]


@pytest.mark.parametrize("case", CASES)
def test_matches_general_kernels(case):
    print("[gpu-case] small PCG %s" % (case,), flush=True)
    A, ctx, _ = system(*case)
    S = A.to_scipy()
    n = S.shape[0]
    rng = np.random.default_rng(n)
    b, x0 = rng.standard_normal(n), rng.standard_normal(n)
    fits = (n <= (1536 if ctx.pattern_info()["box"] else 4096) and S.nnz <= 40960 and
            S.nnz <= 64 * n)
    for precond in (_lib.GH_PRECOND_JACOBI, _lib.GH_PRECOND_NONE):
        x, st = ctx.pcg(b=b, x0=x0, precond=precond, rtol=1e-10)
        assert (ctx.solve_form() == _lib.GH_SOLVE_WORKGROUP) == fits
        y, sy = general(ctx, b=b, x0=x0, precond=precond, rtol=1e-10)
        assert st.converged and sy.converged and abs(st.iterations - sy.iterations) <= 1
        assert np.linalg.norm(b - S @ x) <= 1.01e-10 * np.linalg.norm(b)
        assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
        z, sz = ctx.pcg_noalloc(b=b, x0=x0, precond=precond, rtol=1e-10)
        assert ctx.solve_form() == (_lib.GH_SOLVE_WORKGROUP if fits else _lib.GH_SOLVE_ROWS)
        if fits:  # the same kernel, on other buffers
            np.testing.assert_array_equal(x, z)
        assert np.linalg.norm(x - z) <= 1e-6 * np.linalg.norm(x)
        assert abs(sz.iterations - st.iterations) <= 1
    # the same bits every time
    w, _ = ctx.pcg(b=b, x0=x0, precond=_lib.GH_PRECOND_JACOBI, rtol=1e-10)
    v, _ = ctx.pcg(b=b, x0=x0, precond=_lib.GH_PRECOND_JACOBI, rtol=1e-10)
    np.testing.assert_array_equal(w, v)


def test_limits_and_exact_starts():
    print("[gpu-case] small PCG: iteration limit, exact start, zero b", flush=True)
    A, ctx, _ = system(2, (20, 17))
    S = A.to_scipy()
    b = np.random.default_rng(4).standard_normal(S.shape[0])
    x, st = small(ctx, b=b, rtol=1e-10)
    for maxit in (0, 1, 7):
        got, s1 = small(ctx, b=b, rtol=1e-10, maxit=maxit, raise_on_noconv=False)
        ref, s2 = general(ctx, b=b, rtol=1e-10, maxit=maxit, raise_on_noconv=False)
        assert s1.iterations == s2.iterations == maxit and not s1.converged
        np.testing.assert_allclose(got, ref, rtol=1e-10, atol=1e-14)
        assert abs(s1.rel_residual - s2.rel_residual) <= 1e-10 * s2.rel_residual
    y, s3 = small(ctx, b=b, x0=x, rtol=1e-8)
    assert s3.iterations == 0 and np.array_equal(x, y)
    zero, s4 = small(ctx, b=np.zeros_like(b), rtol=1e-8)
    assert s4.converged and s4.iterations == 0 and not zero.any()
    # a tolerance below what FP64 reaches: restarts run out, as in the general form
    _, s5 = small(ctx, b=b, rtol=1e-30, maxit=5000, raise_on_noconv=False)
    _, s6 = general(ctx, b=b, rtol=1e-30, maxit=5000, raise_on_noconv=False)
    assert not s5.converged and not s6.converged
    # a matrix that is not finite ends like there
    nz, _ = ctx.values_get()
    nz[3] = np.nan
    ctx.values_set(nz)
    _, s7 = small(ctx, b=b, rtol=1e-8, maxit=50, raise_on_noconv=False)
    assert not s7.converged


def test_solve_over_several_launches():
    """Coefficients over fourteen decades, no preconditioner: more iterations than one launch
    runs (8192), so the state goes through the workspace.  In floating point such counts move
    by a percent or two with the rounding of the dot products (5% allowed)."""
    print("[gpu-case] small PCG: several launches", flush=True)
    A, ctx, _ = system(2, (40, 40), spread=4.0)
    S = A.to_scipy()
    b = np.random.default_rng(4).standard_normal(S.shape[0])
    x, st = small(ctx, b=b, rtol=1e-8, maxit=60000, precond=_lib.GH_PRECOND_NONE)
    _, sy = general(ctx, b=b, rtol=1e-8, maxit=60000, precond=_lib.GH_PRECOND_NONE)
    assert st.converged and sy.converged
    assert st.iterations > 8192 and abs(st.iterations - sy.iterations) <= 0.05 * sy.iterations
    assert np.linalg.norm(b - S @ x) <= 1.01e-8 * np.linalg.norm(b)


def test_uneven_rows_are_declined():
    """63 fan meshes, one in each slice of 64 rows: the padded slices would not fit the
    stream; the general kernels solve the system."""
    print("[gpu-case] small PCG: uneven rows", flush=True)
    m, copies = 60, 63
    t = 2 * np.pi * np.arange(m) / m
    one = np.concatenate([[[0, 0, 0]], np.stack([np.cos(t), np.sin(t), 0 * t], 1),
                          [[0, 0, 1.0], [0, 0, -1.0]]])
    r, nx = 1 + np.arange(m), 1 + (np.arange(m) + 1) % m
    cells = np.concatenate([np.stack([0 * r, r, nx, np.full(m, m + 1 + k)], 1) for k in (0, 1)])
    nn = len(one)
    xyz = np.concatenate([one + [5.0 * k, 0, 0] for k in range(copies)])
    cells = np.concatenate([cells + nn * k for k in range(copies)])
    ptrs = (np.arange(len(cells) + 1) * 4 + 1).astype(np.int32)
    cd = (cells + 1).astype(np.int32)
    # the apexes are Dirichlet, so that the matrix is regular
    free = np.ones(len(xyz), bool)
    for k in range(copies):
        free[nn * k + m + 1:nn * k + m + 3] = False
    ids = np.where(free, np.cumsum(free), -np.cumsum(~free))
    cd = ids[cells].astype(np.int32)
    q = G.Quadrature(3, 2, simplex=True)
    shp, grad = G.ReferenceFE(G.lagrangian, G.Float64, 1).tabulate(3, q.coords, simplex=True)
    ctx = _lib.Context(0)
    ctx.mesh_upload(xyz, (cells + 1).astype(np.int32).ravel(), ptrs)
    ctx.space_upload(_lib.GH_REFFE_PK, 1, 1, cd.ravel(), ptrs, int(free.sum()), int((~free).sum()))
    ctx.reffe_tabulation(q.weights, shp, grad)
    ctx.symbolic()
    ctx.assemble()
    assert ctx.nfree <= 4096 and ctx.nnz <= 40960
    x, st = ctx.pcg(rtol=1e-10)
    assert ctx.solve_form() == _lib.GH_SOLVE_ROWS  # declined by the kernel, not by the rule
    y, sy = general(ctx, rtol=1e-10)
    assert st.converged and abs(st.iterations - sy.iterations) <= 1
    np.testing.assert_allclose(x, y, rtol=1e-7, atol=1e-12)
    ctx.close()
