"""The scalar multigrid V-cycle against the same cycle written with dense matrices: transfers by (bi/tri)linear
interpolation, coarse operators by Galerkin products, damped Jacobi sweeps, an exact coarsest solve.

Grids: coarsest systems of 4 to 325 unknowns around the 64 of the blocked inversion's tiles (63, 64, 65, 128, 129), one
plane to enough planes for each number of planes per thread, ragged blocks; 1 to 3 sweeps; box elements (whose matrix
depends on the corners' difference only), a general symmetric element matrix and one that is not symmetric; with and without fixed nodes.

Tolerance: some hundred FP64 operations per entry, amplified by the coarsest solve (condition below 1e5 here): 1e-10 of
the result's largest entry."""
import numpy as np
import pytest
import torch

import pymoto_amd as pm
from pymoto_amd.assembly import poisson_element

pytestmark = pytest.mark.gpu


def interpolation(nc):
    """(2 nc - 1) x nc linear interpolation of one axis with nc coarse nodes."""
    P = np.zeros((2 * nc - 1, nc))
    for i in range(2 * nc - 1):
        P[i, i // 2] += 0.5
        P[i, (i + 1) // 2] += 0.5
    return P


def dense_vcycle(A, nodes, levels, omega, steps, r):
    if levels == 1:
        return np.linalg.solve(A, r)
    dinv = omega / np.diag(A)
    coarse = [(n + 1) // 2 for n in nodes]
    P = np.ones((1, 1))
    for nc, n in zip(coarse, nodes):  # x fastest
        P = np.kron(interpolation(nc) if n > 1 else np.ones((1, 1)), P)
    u = np.zeros_like(r)
    for _ in range(steps):
        u = u + dinv * (r - A @ u)
    u = u + P @ dense_vcycle(P.T @ A @ P, coarse, levels - 1, omega, steps, P.T @ (r - A @ u))
    for _ in range(steps):
        u = u + dinv * (r - A @ u)
    return u


GRIDS = [((2, 2, 0), 2), ((16, 12, 0), 2), ((14, 14, 0), 2), ((24, 8, 0), 2), ((30, 14, 0), 2), ((84, 4, 0), 2),
         ((48, 24, 0), 2), ((40, 24, 0), 3), ((2, 2, 2), 2), ((8, 8, 4), 3), ((12, 8, 16), 2), ((4, 4, 36), 3)]


@pytest.mark.parametrize("kind", ["box", "general", "free", "nonsymmetric"])
@pytest.mark.parametrize("nel,levels", GRIDS)
def test_vcycle_vs_dense(gpu_lib, nel, levels, kind):
    rng = np.random.default_rng(nel[0] + nel[1] + len(kind))
    d = pm.VoxelDomain(*nel)
    nodes = [n + 1 for n in nel]
    E = poisson_element(d)
    if kind == "nonsymmetric":
        G = rng.uniform(-0.1, 0.1, E.shape)
        E = E + G @ G.T + 0.05 * (G - G.T)
    if kind == "general":
        G = rng.uniform(-0.1, 0.1, E.shape)
        E = E + G @ G.T
    if kind == "free":  # no fixed node: a mass term keeps it definite
        E = E + 0.05 * np.eye(E.shape[0])
    bc = None if kind == "free" else np.unique(np.r_[np.arange(0, d.nnodes, nodes[0]), d.nnodes // 2])
    xh = rng.uniform(0.2, 1.0, d.nel)
    K = pm.AssembleGeneral(d, E, bc=bc)(torch.as_tensor(xh).cuda())
    A = np.zeros((d.nnodes, d.nnodes))
    for e, conn in enumerate(np.asarray(d.conn)):
        A[np.ix_(conn, conn)] += float(xh[e]) * E
    if bc is not None:
        A[bc, :] = A[:, bc] = 0.0
        A[bc, bc] = K.grid.bcdiag
    r = rng.standard_normal(d.nnodes)
    steps = 1 + (nel[0] + nel[1]) // 2 % 3
    mg = pm.solvers.build_hierarchy(d, levels, omega=0.6, smooth_steps=steps)
    mg.update(K)
    z = mg.solve(torch.as_tensor(r).cuda()).cpu().numpy()
    ref = dense_vcycle(A, nodes, levels, 0.6, steps, r)
    assert np.abs(z - ref).max() < 1e-10 * np.abs(ref).max()


def axis_interpolate(c, ax):
    """(bi/tri)linear interpolation of one axis: nodes 2 I are copied, those between are means."""
    n = c.shape[ax]
    lo, hi = c.narrow(ax, 0, n - 1), c.narrow(ax, 1, n - 1)
    pairs = torch.stack([lo, 0.5 * (lo + hi)], dim=ax + 1).flatten(ax, ax + 1)
    return torch.cat([pairs, c.narrow(ax, n - 1, 1)], dim=ax)


def axis_restrict(f, ax):
    """Its transpose."""
    n = f.shape[ax]
    even, odd = f.index_select(ax, torch.arange(0, n, 2, device=f.device)), \
        f.index_select(ax, torch.arange(1, n, 2, device=f.device))
    zero = torch.zeros_like(odd.narrow(ax, 0, 1))
    return even + 0.5 * (torch.cat([zero, odd], ax) + torch.cat([odd, zero], ax))


@pytest.mark.parametrize("nel,levels", [((256, 256, 128), 5), ((2048, 2048, 0), 6)])
def test_large_grid_memory_and_coarse_operator(gpu_lib, nel, levels):
    """A grid whose coarse stencils are formed slab by slab: the level-1 product is R^T A R of the fine one (sums of at
    most 27 x 27 products and 27 + 8 terms of the transfers, each good to 2^-53: 1e-12 of the largest entry), and the
    handle takes the stencils (NS doubles per node and 1/(2^D - 1) more), six vectors (r, z, p, q, D^-1, work) on the fine grid
    and four on each coarse one, and 0.3 GB for the coarsest inverse, sums and slabs."""
    d = pm.VoxelDomain(*nel)
    nodes = [n + 1 for n in nel if n]
    g = torch.Generator().manual_seed(1)
    P = pm.AssemblePoisson(d, bc=np.arange(0, 500, 3))(0.1 + torch.rand(d.nel, generator=g, dtype=torch.float64).cuda())
    mg = pm.solvers.build_hierarchy(d, levels, omega=0.5, smooth_steps=2)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    mg._ensure_handle(P)
    used = free - torch.cuda.mem_get_info()[0]
    n, more = P.shape[0], 1.0 / (2 ** d.dim - 1)
    assert used < 8 * n * (3 ** d.dim * (1 + more) + 6 + 4 * more) * 1.02 + 3e8
    mg.update(P)
    shape = [(m + 1) // 2 for m in reversed(nodes)]
    c = torch.randn(shape, generator=g, dtype=torch.float64).cuda()
    f = c
    for ax in range(len(shape)):
        f = axis_interpolate(f, ax)
    f = mg.level_apply(0, f.reshape(-1).contiguous()).reshape(list(reversed(nodes)))
    for ax in range(len(shape)):
        f = axis_restrict(f, ax)
    got = mg.level_apply(1, c.reshape(-1).contiguous()).reshape(shape)
    assert float((got - f).abs().max() / f.abs().max()) < 1e-12
