"""The stencil PCG kernels (box of free Q1 lattice nodes) against the general CSR
kernels on the same system, over box shapes at the edges of their tiles and runs: one
row, fewer rows than a tile, rows of one node, row lengths on both sides of a run's
register share (255) and of the long-row form (512), ragged last tiles.

Both forms form the same products and add a row's entries in the same order; they differ
in the grouping of the dot products only, so the iterates agree to rounding and the
iteration count to one.  The solutions are stopped at a relative residual of 1e-10:
they differ by at most about 1e-10 times the condition of these small systems (< 1e3).
"""
import os

import numpy as np
import pytest

import gridap_hip as G
from gridap_hip import _lib
from gridap_hip import fsai as FS

pytestmark = pytest.mark.gpu

BOXES = [(2, 2, 2), (3, 2, 2), (2, 6, 9), (17, 33, 9), (10, 2, 60), (2, 300, 3), (256, 3, 4),
         (257, 4, 2), (513, 3, 3), (514, 3, 4), (1100, 3, 2), (33, 33, 3)]


def solve(ctx, precond, form):
    old = os.environ.get("GRIDAP_HIP_STENCIL_PCG")
    os.environ["GRIDAP_HIP_STENCIL_PCG"] = form
    try:
        return ctx.pcg(precond=precond, rtol=1e-10, maxit=5000)
    finally:
        if old is None:
            del os.environ["GRIDAP_HIP_STENCIL_PCG"]
        else:
            os.environ["GRIDAP_HIP_STENCIL_PCG"] = old


@pytest.mark.parametrize("part", BOXES)
def test_stencil_and_csr_forms_agree(part):
    print("[gpu-case] stencil PCG %s" % (part,), flush=True)
    rng = np.random.default_rng(sum(part))
    # cubic cells: the condition number is set by the shortest axis
    model = G.CartesianDiscreteModel(tuple(v for n in part for v in (0, n)), part)
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1),
                      dirichlet_tags="boundary")
    dx = G.Measure(G.Triangulation(model), 2)
    k = G.CellField(np.exp(rng.normal(size=model.num_cells())), None)
    op = G.AffineFEOperator(lambda u, v: G.integrate(k * G.inner(G.gradient(v), G.gradient(u)), dx),
                            lambda v: G.integrate(1.0 * v, dx), G.TrialFESpace(V), V)
    ctx = op.assem.ctx
    assert ctx.pattern_info()["box"] == 1
    A, b = op.get_matrix().to_scipy(), op.get_vector()
    FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).attach(ctx)
    for precond in (_lib.GH_PRECOND_NONE, _lib.GH_PRECOND_JACOBI, _lib.GH_PRECOND_FSAI):
        x, st = solve(ctx, precond, "1")
        assert ctx.solve_form() == _lib.GH_SOLVE_STENCIL
        y, sy = solve(ctx, precond, "0")
        assert ctx.solve_form() == _lib.GH_SOLVE_ROWS
        assert abs(st.iterations - sy.iterations) <= 1
        assert np.linalg.norm(b - A @ x) <= 1e-10 * np.linalg.norm(b)
        assert np.linalg.norm(x - y) <= 1e-7 * np.linalg.norm(y)
