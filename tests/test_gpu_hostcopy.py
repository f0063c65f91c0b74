"""Host arrays through the library's pinned staging: sizes around a chunk (1 MiB) and the
four chunks in flight, more calls at once than idle buffers are kept, threads with
contexts of their own, and without pinned memory.  The copies move bytes: the comparison is exact."""
import threading

import numpy as np
import pytest

import gridap_hip as G
from gridap_hip import _lib

pytestmark = pytest.mark.gpu


def lattice(n, seed):
    """A 2-D Q1 context with about n free dofs (all nodes free)."""
    ny = 3
    nx = max(2, n // (ny + 1) - 1)
    model = G.CartesianDiscreteModel((0, 1, 0, 1), (nx, ny))
    V = G.TestFESpace(model, G.ReferenceFE(G.lagrangian, G.Float64, 1))
    q = G.Quadrature(2, 2)
    shp, grad = V.reffe.tabulate(2, q.coords)
    cd = V.get_cell_dof_ids()
    ptrs = (np.arange(len(cd) + 1, dtype=np.int64) * 4 + 1).astype(np.int32)
    ctx = _lib.Context(0)
    ctx.mesh_cartesian(model.origin, model.sizes, model.partition)
    ctx.space_upload(_lib.GH_REFFE_QK, 1, 1, cd.ravel(), ptrs, V.nfree, 0)
    ctx.reffe_tabulation(q.weights, shp, grad)
    ctx.symbolic()
    ctx.coef_upload(np.exp(np.random.default_rng(seed).normal(size=model.num_cells())))
    ctx.assemble()
    return ctx


# doubles: one chunk holds 131,072; nzval has about eight entries a dof
@pytest.mark.parametrize("n", [12, 16_380, 16_390, 131_060, 131_080, 131_072 * 4 + 4, 700_000])
def test_values_round_trip(n):
    print("[gpu-case] staged copies, %d dofs" % n, flush=True)
    ctx = lattice(n, n)
    rng = np.random.default_rng(n)
    nz, b = rng.standard_normal(ctx.nnz), rng.standard_normal(ctx.nfree)
    ctx.values_set(nz, b)
    gz, gb = ctx.values_get()
    np.testing.assert_array_equal(gz, nz)
    np.testing.assert_array_equal(gb, b)
    cp, rv = ctx.pattern_get()
    assert cp[0] == 1 and cp[-1] == ctx.nnz + 1 and len(rv) == ctx.nnz
    assert rv.min() == 1 and rv.max() == ctx.nfree
    # sorted rows in every column: a chunk out of place would break the order somewhere
    inside = np.ones(ctx.nnz - 1, dtype=bool)
    inside[cp[1:-1] - 2] = False
    assert np.all(np.diff(rv)[inside] > 0)
    ctx.close()


@pytest.mark.parametrize("n", [12, 131_072 * 4 + 4])
def test_without_pinned_memory(n, monkeypatch):
    """Pinning refused (GRIDAP_HIP_PINNED=0 answers for the runtime): the same bytes through
    direct copies, and the solve that is paced by a pinned word reads back instead."""
    print("[gpu-case] direct copies, %d dofs" % n, flush=True)
    monkeypatch.setenv("GRIDAP_HIP_SMALL_PCG", "0")
    got = []
    for pinned in ("1", "0"):
        monkeypatch.setenv("GRIDAP_HIP_PINNED", pinned)
        ctx = lattice(n, n)
        nz, b = ctx.values_get()
        nz = nz.copy()
        cp, rv = ctx.pattern_get()
        nz[np.flatnonzero(rv - 1 == np.repeat(np.arange(ctx.nfree), np.diff(cp)))] += 1.0
        ctx.values_set(nz, np.random.default_rng(n).standard_normal(ctx.nfree))
        x, st = ctx.pcg(rtol=1e-10)
        got.append((cp, rv, *ctx.values_get(), x, ctx.spmv(x), st.iterations))
        ctx.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


def test_threads_with_their_own_contexts():
    print("[gpu-case] staged copies, 12 threads", flush=True)
    ctxs = [lattice(40_000 + 4000 * k, k) for k in range(12)]
    bad = []

    def work(ctx, seed):
        rng = np.random.default_rng(seed)
        for _ in range(5):
            nz, b = rng.standard_normal(ctx.nnz), rng.standard_normal(ctx.nfree)
            ctx.values_set(nz, b)
            gz, gb = ctx.values_get()
            if not (np.array_equal(gz, nz) and np.array_equal(gb, b)):
                bad.append(seed)

    threads = [threading.Thread(target=work, args=(c, k)) for k, c in enumerate(ctxs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for c in ctxs:
        c.close()
