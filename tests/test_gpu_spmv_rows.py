"""The CSR row kernels (SpMV, and the general PCG that reads the same rows) over every row
shape they are chosen for: mean row lengths of 1 to 190, rows longer than one turn of
their lanes, one row, and sizes off the rows-per-workgroup count.

y is compared with scipy's product of the same stored values: both add at most a few
hundred products of a row in FP64, in different orders, so they agree to
(row length) x 2^-53 of Σ|a||x|, below 1e-13.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import gridap_hip as G
from gridap_hip import _lib

pytestmark = pytest.mark.gpu


def _operator(D, part, order, ncomp, tags):
    model = G.CartesianDiscreteModel((0, 1) * D, part)
    T = G.VectorValue[D, G.Float64] if ncomp > 1 else G.Float64
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, T, order), dirichlet_tags=tags)
    dx = G.Measure(G.Triangulation(model), 2 * order)
    if ncomp > 1:
        s = G.IsotropicStress(1.0, 0.3)
        a = lambda u, v: G.integrate(G.inner(G.ε(v), s(G.ε(u))), dx)
    else:
        a = lambda u, v: G.integrate(G.inner(G.gradient(v), G.gradient(u)), dx)
    assem = G.SparseMatrixAssembler(G.TrialFESpace(V), V)
    return assem.ctx, G.assemble_matrix(a, assem, G.TrialFESpace(V), V), assem


CASES = [
    (2, (2, 2), 1, 1, "boundary"),          # one row of one entry
    (2, (9, 7), 1, 1, "boundary"),          # rows of 4 to 9: four lanes
    (2, (131, 3), 1, 1, "tag_1"),
    (3, (7, 5, 6), 1, 1, ["tag_21"]),       # 8 to 27: eight lanes
    (2, (12, 9), 2, 1, "boundary"),         # scalar Q2 in 2-D
    (3, (5, 4, 3), 2, 1, "boundary"),       # 27 to 125: sixteen lanes
    (2, (6, 5), 2, 2, "boundary"),          # vector Q2 in 2-D
    (3, (3, 2, 3), 2, 3, ["tag_25"]),       # up to 375: thirty-two lanes, two turns
]


@pytest.mark.parametrize("case", CASES)
def test_row_kernels(case, monkeypatch):
    monkeypatch.setenv("GRIDAP_HIP_STENCIL_PCG", "0")  # the CSR kernels, whatever the size
    print("[gpu-case] CSR rows %s" % (case,), flush=True)
    _, A, assem = _operator(*case)
    S = A.to_scipy()
    rng = np.random.default_rng(3)
    x = rng.standard_normal(S.shape[0])
    y = assem.ctx.spmv(x)
    assert np.all(np.abs(y - S @ x) <= 1e-13 * (abs(S) @ np.abs(x)))
    b = rng.standard_normal(S.shape[0])
    for precond in (_lib.GH_PRECOND_NONE, _lib.GH_PRECOND_JACOBI):
        u, st = assem.ctx.pcg(b=b, precond=precond, rtol=1e-10)
        assert assem.ctx.solve_form() == _lib.GH_SOLVE_ROWS
        assert np.linalg.norm(b - S @ u) <= 1.01e-10 * np.linalg.norm(b), st.rel_residual


@pytest.mark.parametrize("case", CASES)
def test_infinite_entries(case):
    """One ±Inf in x: the rows that hold its column are infinite (NaN where the stored value
    is 0), whatever their length is to the turn of their lanes."""
    print("[gpu-case] CSR rows, infinite entry %s" % (case,), flush=True)
    _, A, assem = _operator(*case)
    S = A.to_scipy().tocsr()
    rng = np.random.default_rng(5)
    for j in sorted({0, S.shape[0] - 1, *rng.integers(S.shape[0], size=6)}):
        x = rng.standard_normal(S.shape[0])
        x[j] = rng.choice([np.inf, -np.inf])
        y, ref = assem.ctx.spmv(x), S @ x
        fin = np.isfinite(ref)
        assert not fin.all()
        np.testing.assert_array_equal(y[~fin], ref[~fin])
        x[j] = 0.0
        assert np.all(np.abs(y[fin] - ref[fin]) <= 1e-13 * (abs(S) @ np.abs(x))[fin])


def test_one_long_row_among_short_ones():
    """A vertex shared by 300 tetrahedra: its row holds every column, the others seven."""
    print("[gpu-case] CSR rows, fan mesh", flush=True)
    n = 150
    t = 2 * np.pi * np.arange(n) / n
    xyz = np.concatenate([[[0, 0, 0]], np.stack([np.cos(t), np.sin(t), 0 * t], 1), [[0, 0, 1.0]],
                          [[0, 0, -1.0]]])
    r = 1 + np.arange(n)
    nxt = 1 + (np.arange(n) + 1) % n
    cells = np.concatenate([np.stack([0 * r, r, nxt, np.full(n, n + 1 + k)], 1) for k in (0, 1)])
    ptrs = (np.arange(len(cells) + 1) * 4 + 1).astype(np.int32)
    cd = (cells + 1).astype(np.int32)
    q = G.Quadrature(3, 2, simplex=True)
    shp, grad = G.ReferenceFE(G.lagrangian, G.Float64, 1).tabulate(3, q.coords, simplex=True)
    ctx = _lib.Context(0)
    ctx.mesh_upload(xyz, cd.ravel(), ptrs)
    ctx.space_upload(_lib.GH_REFFE_PK, 1, 1, cd.ravel(), ptrs, n + 3, 0)
    ctx.reffe_tabulation(q.weights, shp, grad)
    ctx.symbolic()
    ctx.assemble(_lib.GH_FORM_DIFFUSION, _lib.GH_PREC_FP64)
    nz, _ = ctx.values_get()
    cp, rv = ctx.pattern_get()
    S = sp.csc_matrix((nz, rv - 1, cp - 1), shape=(n + 3, n + 3))
    x = np.random.default_rng(1).standard_normal(n + 3)
    assert np.all(np.abs(ctx.spmv(x) - S @ x) <= 1e-13 * (abs(S) @ np.abs(x)))
    ctx.close()
