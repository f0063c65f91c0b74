"""The training step of the learned FSAI at the edges of its tiles and batches, against
an FP64 PyTorch evaluation of the same step (needs an MI355X).

The device keeps activations, their gradients and the weight sums in FP32 (FP64 from 256
cells on: between a workgroup's runs of four tiles, and where the partials of the workgroups
meet); weights are the same BF16 values on both sides.  A contraction has at most 64 terms
and a weight sum in FP32 at most 256, so a gradient carries a few 1e-7 relative; the network is three layers deep and the pattern gradient
is rounded to FP32 once: 2e-5 (relative L2 per layer) bounds it, and 1e-6 the loss, whose
factor entries are rounded to FP32.
"""
import numpy as np
import pytest
import torch

import fsai_oracle as F
from gridap_hip import _lib
from test_gpu_fsai import make_context, random_params

pytestmark = pytest.mark.gpu

# cells: fewer than a tile, one tile, one past it, ragged last tile, more tiles than
# workgroups of the backward (256 x 64 cells)
CASES = [((2, 2, 2), 1), ((4, 4, 4), 2), ((5, 13, 1), 3), ((5, 13, 2), 3), ((13, 11, 9), 4),
         ((9, 8, 7), 7), ((27, 26, 25), 5)]


def reference(ctx, part, kappa, params, seed, m):
    """(network output, loss, weight gradient) in FP64, cell by cell."""
    C = int(np.prod(part))
    nn = [p + 1 for p in part]
    c = np.arange(C)
    x, y, z = c % part[0], (c // part[0]) % part[1], c // (part[0] * part[1])
    node = np.stack([(x + (a & 1)) + nn[0] * ((y + (a >> 1 & 1)) + nn[1] * (z + (a >> 2)))
                     for a in range(8)], 1)
    n = np.arange(int(np.prod(nn)))
    ijk = (n % nn[0], (n // nn[0]) % nn[1], n // (nn[0] * nn[1]))
    free = np.all([(v > 0) & (v < p) for v, p in zip(ijk, part)], axis=0)
    dof = np.where(free, np.cumsum(free) - 1, -1)[node]
    N = int(free.sum())
    at = torch.as_tensor(np.where(dof >= 0, dof, N))
    cp, rv = ctx.pattern_get()
    nz, _ = ctx.values_get()
    A = torch.sparse_csr_tensor(torch.as_tensor(cp - 1), torch.as_tensor(rv - 1),
                                torch.as_tensor(nz), (N, N))
    diag = torch.as_tensor(nz[np.flatnonzero(rv - 1 == np.repeat(np.arange(N), np.diff(cp)))])
    s = diag ** -0.5
    local = lambda v: torch.cat([v, v.new_zeros(1)])[at]
    total = lambda v: torch.zeros(N + 1, dtype=torch.float64).index_add(
        0, at.reshape(-1), v.reshape(-1))[:N]
    w = torch.as_tensor(params).to(torch.bfloat16).double().requires_grad_(True)
    cut, k = [], 0
    for shape in ((64, 10), (64,), (64, 64), (64,), (64, 64), (64,), (36, 64), (36,)):
        cut.append(w[k:k + int(np.prod(shape))].reshape(shape))
        k += int(np.prod(shape))
    h = torch.as_tensor(ctx.fsai_get()["feat"][:, :10].astype(np.float64))
    for i in range(0, 6, 2):
        h = torch.nn.functional.gelu(h @ cut[i].T + cut[i + 1])
    out = h @ cut[6].T + cut[7]
    L = torch.zeros(C, 8, 8, dtype=torch.float64)
    pairs = [(a, b) for a in range(8) for b in range(a)]
    L[:, [a for a, _ in pairs], [b for _, b in pairs]] = out[:, 8:]
    d = total(out[:, :8]).exp()
    mul = lambda M, v: total((M * local(v)[:, None, :]).sum(-1))
    loss = 0.0
    for p in range(m):
        v = torch.as_tensor(F.rademacher(seed, p, N))
        t = s * (d * v + mul(L.transpose(1, 2), v))
        q = A @ t
        r = v - (d * (s * q) + mul(L, s * q))
        loss = loss + r @ r
    loss = loss / (m * N)
    (g,) = torch.autograd.grad(loss, w)
    return out.detach().numpy(), float(loss.detach()), g.numpy()


# W1, b1, W2, b2, W3, b3, W4, b4 in the flat parameters
LAYERS = ((0, 640), (640, 704), (704, 4800), (4800, 4864), (4864, 8960), (8960, 9024),
          (9024, 11328), (11328, 11364))


@pytest.mark.parametrize("part,bounds", [
    # what kernels with FP32 sums of 256 cells for every partial had on this very input
    ((64, 64, 64), (3.6e-8, 2.9e-8, 3.3e-8, 3.1e-8, 3.5e-8, 2.9e-8, 4.1e-8, 4.2e-8)),
    # one FP32 rounding of every gradient (with sums of 3456 cells W2 had 6.7e-8)
    ((96, 96, 96), (2.0 ** -24,) * 8)])
def test_many_tiles_a_workgroup(part, bounds):
    """16 and 54 tiles a workgroup of the backward: the error of the gradients does not grow
    with the mesh."""
    print("[gpu-case] fsai training step %s, many tiles" % (part,), flush=True)
    kappa = np.exp(np.random.default_rng(2).normal(size=int(np.prod(part))))
    ctx = make_context(part, kappa)
    params = random_params(2, scale4=0.05)
    ctx.mlp_set(params)
    ctx.fsai_train_step(2, 4321, 0.0)
    got = ctx.fsai_get()["grad"]
    _, _, g = reference(ctx, part, kappa, params, 4321, 2)
    for (lo, hi), bound in zip(LAYERS, bounds):
        assert np.linalg.norm(got[lo:hi] - g[lo:hi]) <= bound * np.linalg.norm(g[lo:hi]), lo
    ctx.close()


@pytest.mark.parametrize("part,probes", CASES)
def test_step_matches_fp64(part, probes):
    print("[gpu-case] fsai training step %s, %d probes" % (part, probes), flush=True)
    if 1 in part:
        part = tuple(max(2, p) for p in part)
    kappa = np.exp(np.random.default_rng(probes).normal(size=int(np.prod(part))))
    ctx = make_context(part, kappa)
    params = random_params(probes, scale4=0.05)
    ctx.mlp_set(params)
    loss = ctx.fsai_train_step(probes, 4321, 0.0)
    got = ctx.fsai_get()
    out, ref, g = reference(ctx, part, kappa, params, 4321, probes)
    assert np.abs(got["yout"][:, :36] - out).max() <= 1e-5 * np.abs(out).max()
    assert abs(loss - ref) <= 1e-6 * ref
    for lo, hi in LAYERS:
        err = np.linalg.norm(got["grad"][lo:hi] - g[lo:hi]) / np.linalg.norm(g[lo:hi])
        assert err <= 2e-5, (lo, err)
    # lr = 0 leaves the solver's factor of these weights; a step leaves none
    ctx.fsai_factor_get()
    ctx.fsai_train_step(probes, 1, 1e-3)
    assert np.abs(ctx.mlp_get() - params).max() > 0
    with pytest.raises(_lib.GridapHipError):
        ctx.fsai_factor_get()
    ctx.close()
