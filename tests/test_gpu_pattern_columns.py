"""The pattern built column by column (spaces that keep contribution lists) on columns at the
edges of its sort: one cell, 64 candidates and one cell more, just under its limit of 2048
and past it (global sort), several components of the mesh in one column count, Dirichlet
rows, against the pattern and the P1 stiffness matrix formed on the host (needs an MI355X).

Values: sums of at most 700 FP64 element entries, each with a relative error of a few eps."""
import numpy as np
import pytest
import scipy.sparse as sp

import gridap_hip as G
from gridap_hip import _lib

pytestmark = pytest.mark.gpu


def fan(m):
    """m-gon around an axis of two tetrahedra rings: the centre touches 2 m cells."""
    t = 2 * np.pi * np.arange(m) / m
    xyz = np.concatenate([[[0, 0, 0]], np.stack([np.cos(t), np.sin(t), 0 * t], 1),
                          [[0, 0, 1.0], [0, 0, -1.0]]])
    r, nx = 1 + np.arange(m), 1 + (np.arange(m) + 1) % m
    up = np.stack([0 * r, r, nx, np.full(m, m + 1)], 1)
    down = np.stack([0 * r, nx, r, np.full(m, m + 2)], 1)
    return xyz, np.concatenate([up, down])


@pytest.mark.parametrize("m", [3, 8, 9, 127, 128, 129, 255, 256, 257, 350])
@pytest.mark.parametrize("fixed", ["apexes", "ring", "none"])
def test_fan_pattern_and_matrix(m, fixed):
    print("[gpu-case] pattern columns fan %d %s" % (m, fixed), flush=True)
    xyz, cells = fan(m)
    free = np.ones(len(xyz), bool)
    if fixed == "apexes":
        free[m + 1:] = False
    if fixed == "ring":
        free[1:m + 1:2] = False
    ids = np.where(free, np.cumsum(free), -np.cumsum(~free))
    ptrs = (np.arange(len(cells) + 1) * 4 + 1).astype(np.int32)
    cd = ids[cells].astype(np.int32)
    q = G.Quadrature(3, 2, simplex=True)
    shp, grad = G.ReferenceFE(G.lagrangian, G.Float64, 1).tabulate(3, q.coords, simplex=True)
    ctx = _lib.Context(0)
    ctx.mesh_upload(xyz, (cells + 1).astype(np.int32).ravel(), ptrs)
    ctx.space_upload(_lib.GH_REFFE_PK, 1, 1, cd.ravel(), ptrs, int(free.sum()), int((~free).sum()))
    ctx.reffe_tabulation(q.weights, shp, grad)
    ctx.symbolic()
    ctx.assemble()
    # ∫ ∇φa·∇φb on a tetrahedron
    J = xyz[cells[:, 1:]] - xyz[cells[:, :1]]
    g = np.linalg.inv(J).transpose(0, 2, 1)
    g = np.concatenate([-g.sum(1, keepdims=True), g], 1)
    K = np.matmul(g, g.transpose(0, 2, 1)) * (np.abs(np.linalg.det(J)) / 6)[:, None, None]
    i, j = np.repeat(cells, 4, 1), np.tile(cells, (1, 4))
    ref = sp.coo_matrix((K.ravel(), (i.ravel(), j.ravel())), shape=(len(xyz),) * 2).tocsc()
    ones = sp.coo_matrix((np.ones(i.size), (i.ravel(), j.ravel())), shape=ref.shape).tocsc()
    ref, ones = ref[free][:, free], ones[free][:, free]
    ref.sort_indices()
    ones.sort_indices()
    cp, rv = ctx.pattern_get()
    np.testing.assert_array_equal(np.asarray(cp) - 1, ones.indptr)
    np.testing.assert_array_equal(np.asarray(rv) - 1, ones.indices)
    nz, _ = ctx.values_get()
    A = sp.csc_matrix((nz, ones.indices, ones.indptr), shape=ones.shape)
    assert abs(A - ref).max() <= 1e-13 * abs(ref).max()
    ctx.close()
