"""The solve of a box system in one launch of resident workgroups against the launched
stencil kernels on the same system: fewer rows than a workgroup, rows at the edges of the
workgroups (512 and 1024 rows) and of their number (256), long and short lattice rows, the
largest systems it takes and ones past them, restarts, limits, a solve over several launches
and calls from two threads at once (needs an MI355X).

Both form the same products and add a row's entries in the same order; they differ in the
grouping of the dot products only: after 20 iterations the iterates agree to rounding
(20 iterations x condition 1e4 x 2 eps = 1e-10), and the
solutions, stopped at 1e-10, to 1e-10 times the condition (below 1e4 here).  Rounding acts
on CG like a small spread of the eigenvalues (Greenbaum 1989), whose effect on the count
grows with the count: one iteration, or 1% in solves of hundreds."""
import os
import threading

import numpy as np
import pytest

import gridap_hip as G
from gridap_hip import _lib
from gridap_hip import fsai as FS

pytestmark = pytest.mark.gpu

PRECONDS = (_lib.GH_PRECOND_NONE, _lib.GH_PRECOND_JACOBI, _lib.GH_PRECOND_FSAI)


@pytest.fixture(autouse=True)
def no_small(monkeypatch):
    monkeypatch.setenv("GRIDAP_HIP_SMALL_PCG", "0")


def system(part, spread=1.0):
    # cubic cells: the condition number is set by the shortest axis
    model = G.CartesianDiscreteModel(tuple(v for n in part for v in (0, n)), part)
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1),
                      dirichlet_tags="boundary")
    dx = G.Measure(G.Triangulation(model), 2)
    rng = np.random.default_rng(sum(part))
    k = G.CellField(np.exp(rng.normal(0, spread, model.num_cells())), None)
    op = G.AffineFEOperator(lambda u, v: G.integrate(k * G.inner(G.gradient(v), G.gradient(u)), dx),
                            lambda v: G.integrate(1.0 * v, dx), G.TrialFESpace(V), V)
    assert op.assem.ctx.pattern_info()["box"] == 1
    return op, op.assem.ctx


def launched(monkeypatch, ctx, **kw):
    with monkeypatch.context() as m:
        m.setenv("GRIDAP_HIP_RESIDENT_PCG", "0")
        r = ctx.pcg(**kw)
    assert ctx.solve_form() == _lib.GH_SOLVE_STENCIL
    return r


def resident(ctx, **kw):
    r = ctx.pcg(**kw)
    assert ctx.solve_form() == _lib.GH_SOLVE_RESIDENT
    return r


def fits(part, precond):
    """Rows a workgroup (256 compute units): at most 1024 with FSAI, else what LDS holds of
    the vector's three runs and 32 values of each row past 1024."""
    m0, n = part[0] - 1, int(np.prod([p - 1 for p in part]))
    rows = max(-(-(-(-n // 256)) // 64) * 64, 512)
    if precond == _lib.GH_PRECOND_FSAI:
        return rows <= 1024 and 7 * (rows + 2 * m0 + 2) <= 150 * 128
    return max(3 * (rows + 2 * m0 + 2), 3456) + 32 * max(rows - 1024, 0) <= 150 * 128


# free rows: 1, 2, 40, 512, 528, 8 long lattice rows, 16 x 15 x 1025, 64 x 64 x 63 = 258,048
# (1024 a workgroup), 64^3 = 262,144, 65 x 64 x 63 = 262,080, 64 x 65 x 64 past one row a
# thread (FSAI's largest), 71 x 70 x 69 and 72 x 70 x 72 up to the most that LDS holds, and
# 74 x 72 x 72 past it
PARTS = [(2, 2, 2), (3, 2, 2), (2, 6, 9), (33, 17, 2), (34, 17, 2), (514, 3, 3), (1100, 4, 5),
         (17, 16, 1026), (65, 65, 64), (65, 65, 65), (66, 65, 64), (65, 66, 65),
         (72, 71, 70), (73, 71, 73), (75, 73, 73)]


@pytest.mark.parametrize("part", PARTS)
def test_matches_launched_kernels(part, monkeypatch):
    print("[gpu-case] resident PCG %s" % (part,), flush=True)
    op, ctx = system(part)
    A, b = op.get_matrix().to_scipy(), op.get_vector()
    x0 = np.random.default_rng(1).standard_normal(len(b))
    FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).attach(ctx)
    for precond in PRECONDS:
        kw = dict(x0=x0, precond=precond, rtol=1e-10, maxit=5000)
        x, st = ctx.pcg(**kw)
        assert ctx.solve_form() == (_lib.GH_SOLVE_RESIDENT if fits(part, precond)
                                    else _lib.GH_SOLVE_STENCIL)
        y, sy = launched(monkeypatch, ctx, **kw)
        assert st.converged and sy.converged
        assert abs(st.iterations - sy.iterations) <= max(1, 0.01 * sy.iterations)
        assert np.linalg.norm(b - A @ x) <= 1.01e-10 * np.linalg.norm(b)
        assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
        if precond != _lib.GH_PRECOND_FSAI:  # (FSAI at its limit goes on with Jacobi)
            few = dict(kw, maxit=20, raise_on_noconv=False)
            u, v = ctx.pcg(**few)[0], launched(monkeypatch, ctx, **few)[0]
            assert np.linalg.norm(u - v) <= 1e-10 * np.linalg.norm(v)
        z, _ = ctx.pcg(**kw)  # the same bits every time
        np.testing.assert_array_equal(x, z)


def test_limits_and_exact_starts(monkeypatch):
    print("[gpu-case] resident PCG: limits", flush=True)
    op, ctx = system((20, 18, 17))
    b = op.get_vector()
    FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).attach(ctx)
    for precond in PRECONDS:
        x, _ = resident(ctx, precond=precond, rtol=1e-10)
        for maxit in (0, 1, 5):
            kw = dict(precond=precond, rtol=1e-10, maxit=maxit, raise_on_noconv=False)
            got, s1 = resident(ctx, **kw)
            ref, s2 = launched(monkeypatch, ctx, **kw)
            # (FSAI that ends at its limit is followed by as many Jacobi iterations)
            assert s1.iterations == s2.iterations and not s1.converged
            assert s1.iterations == maxit * (2 if precond == _lib.GH_PRECOND_FSAI else 1)
            np.testing.assert_allclose(got, ref, rtol=1e-10, atol=1e-13 * abs(ref).max())
        y, s3 = resident(ctx, x0=x, precond=precond, rtol=1e-8)
        assert s3.iterations == 0 and np.array_equal(x, y)
        zero, s4 = resident(ctx, b=np.zeros_like(b), precond=precond, rtol=1e-8)
        assert s4.converged and s4.iterations == 0 and not zero.any()
        # below what FP64 reaches: the restarts run out
        _, s5 = resident(ctx, precond=precond, rtol=1e-30, maxit=3000, raise_on_noconv=False)
        assert not s5.converged
    nz, _ = ctx.values_get()
    nz[3] = np.nan
    ctx.values_set(nz)
    _, s6 = resident(ctx, rtol=1e-8, maxit=50, raise_on_noconv=False)
    assert not s6.converged


def test_solve_over_several_launches(monkeypatch):
    """Coefficients over many decades, no preconditioner: more iterations than one launch
    runs (2048).  In floating point such counts move by a percent or two with the rounding
    of the dot products (5% allowed)."""
    print("[gpu-case] resident PCG: several launches", flush=True)
    op, ctx = system((40, 40, 2), spread=4.0)
    A, b = op.get_matrix().to_scipy(), op.get_vector()
    kw = dict(rtol=1e-8, maxit=60000, precond=_lib.GH_PRECOND_NONE)
    x, st = resident(ctx, **kw)
    _, sy = launched(monkeypatch, ctx, **kw)
    assert st.converged and sy.converged
    assert st.iterations > 2048 and abs(st.iterations - sy.iterations) <= 0.05 * sy.iterations
    assert np.linalg.norm(b - A @ x) <= 1.01e-8 * np.linalg.norm(b)


# one row a thread and rows past it in LDS
@pytest.mark.parametrize("part", [(20, 18, 17), (66, 65, 66)])
def test_pauses_leave_no_trace(part, monkeypatch):
    """A launch that ends after every iteration, or every third, gives the bits of an
    undivided solve, also where it ends right after a restart: the tolerance is one that
    only the recurrence's r reaches, so that every solve restarts until it may no more."""
    print("[gpu-case] resident PCG: pauses %s" % (part,), flush=True)
    _, ctx = system(part)
    FS.LearnedFSAI.load(FS.DEFAULT_WEIGHTS).attach(ctx)
    for precond in PRECONDS:
        if not fits(part, precond):
            continue
        kw = dict(precond=precond, rtol=1e-30, maxit=1200, raise_on_noconv=False)
        x, st = resident(ctx, **kw)
        for pause in ("1", "3"):
            with monkeypatch.context() as m:
                m.setenv("GRIDAP_HIP_RESIDENT_PAUSE", pause)
                y, sy = resident(ctx, **kw)
            assert (st.iterations, st.rel_residual) == (sy.iterations, sy.rel_residual)
            np.testing.assert_array_equal(x, y)


def test_given_up_solves_are_counted(monkeypatch):
    """A solve whose first, second or fourth launch gives up goes on with the launched kernels
    from the iterate it had: iterations, limit and time cover both."""
    print("[gpu-case] resident PCG: given up", flush=True)
    _, ctx = system((20, 18, 17))
    for precond in PRECONDS[:2]:  # (FSAI that ends at a limit goes on with Jacobi)
        for launch, limit in ((0, 5000), (1, 5000), (3, 5000), (0, 9), (1, 9), (3, 9)):
            done = 2 * launch
            kw = dict(precond=precond, rtol=1e-10, raise_on_noconv=False)
            first, _ = resident(ctx, **kw, maxit=done)
            ref, s1 = launched(monkeypatch, ctx, **kw, x0=first, maxit=limit - done)
            with monkeypatch.context() as m:
                m.setenv("GRIDAP_HIP_RESIDENT_PAUSE", "2")
                m.setenv("GRIDAP_HIP_RESIDENT_GIVE_UP", str(launch))
                x, st = ctx.pcg(**kw, maxit=limit)
            assert ctx.solve_form() == _lib.GH_SOLVE_STENCIL
            assert st.iterations == done + s1.iterations <= limit
            assert st.converged == s1.converged == (limit == 5000)
            np.testing.assert_array_equal(x, ref)
    # 40 launches of an iteration and a read-back each, then one launched iteration
    _, s1 = launched(monkeypatch, ctx, rtol=1e-10, maxit=1, raise_on_noconv=False)
    monkeypatch.setenv("GRIDAP_HIP_RESIDENT_PAUSE", "1")
    monkeypatch.setenv("GRIDAP_HIP_RESIDENT_GIVE_UP", "40")
    _, st = ctx.pcg(rtol=1e-10, maxit=41, raise_on_noconv=False)
    assert st.iterations == 41 and st.device_ms > 3 * s1.device_ms


def test_two_threads():
    """Two contexts solve at once: whichever finds the device's turn taken runs the launched
    kernels; both are right."""
    print("[gpu-case] resident PCG: two threads", flush=True)
    systems = [system((33, 30, 31)), system((40, 28, 26))]
    refs = [resident(ctx, rtol=1e-10)[0] for _, ctx in systems]
    err, forms = [None, None], set()

    def work(k):
        for _ in range(4):
            x, st = systems[k][1].pcg(rtol=1e-10)
            forms.add(systems[k][1].solve_form())
            e = np.linalg.norm(x - refs[k]) / np.linalg.norm(refs[k])
            err[k] = max(err[k] or 0.0, e if st.converged else np.inf)

    ts = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert max(err) <= 1e-6
    assert _lib.GH_SOLVE_RESIDENT in forms  # the first to find the turn free
    assert forms <= {_lib.GH_SOLVE_RESIDENT, _lib.GH_SOLVE_STENCIL}
