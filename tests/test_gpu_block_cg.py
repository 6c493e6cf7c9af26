"""Block CG at every number of columns that selects other kernels (1, 2, 3, 4, 5, 8 and 9: two blocks, the second of
one column), on grids with fewer rows than one block of threads and with rows left over, in 2D and 3D, with and
without captured iterations, restarts and a start vector, and with dependent columns at either end of the block.

A solution is checked by its true residual (the operator's product, FP64): the recursion stops at 1e-10 and is
restarted from the true residual, and the residual of a 1e-10 solution of these small operators carries rounding of
about 1e-13, so 2e-10 bounds it."""
import numpy as np
import pytest
import torch

import pymoto_amd as pm
from oracle import problems

pytestmark = pytest.mark.gpu


def problem(nel, k, seed):
    g = torch.Generator().manual_seed(seed)
    d = pm.VoxelDomain(*nel)
    nx, ny = nel[0] + 1, nel[1] + 1
    if nel[2]:
        bc = problems.cantilever3d(*nel)[0]
    else:
        bc = np.array([2 * j * nx + c for j in range(ny) for c in range(2)])
    x = (0.2 + 0.8 * torch.rand(d.nel, generator=g, dtype=torch.float64)).cuda()
    K = pm.AssembleStiffness(d, bc=bc)(x)
    B = torch.randn(K.shape[0], k, generator=g, dtype=torch.float64)
    B[torch.as_tensor(np.asarray(bc, dtype=np.int64)), :] = 0.0
    return d, K, B.cuda()


def true_residual(K, X, B):
    return max(float((K.residual(B[:, j].contiguous(), X[:, j].contiguous())).norm() / B[:, j].norm())
               for j in range(B.shape[1]))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("k", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("nel,levels", [((8, 4, 0), 2), ((4, 4, 4), 2), ((20, 12, 4), 3), ((88, 80, 0), 4)])
def test_block_columns(gpu_lib, nel, levels, k, prec):
    d, K, B = problem(nel, k, 3 * k + nel[0])
    mg = pm.solvers.build_hierarchy(d, levels, omega=0.4, smooth_steps=2, precision=prec)
    for graph, restart in ((False, 3), (True, 50)):
        cg = pm.solvers.CG(preconditioner=mg, tol=1e-10, maxit=300, restart=restart, graph=graph)
        cg.update(K)
        X = cg.solve(B)
        assert cg.iterations < 300 and true_residual(K, X, B) < 2e-10
        Y = cg.solve(B, x0=0.5 * X)
        assert cg.iterations < 300 and true_residual(K, Y, B) < 2e-10


@pytest.mark.parametrize("k", [2, 3, 4, 6, 8])
def test_dependent_columns(gpu_lib, k):
    d, K, B = problem((12, 8, 4), k, k)
    B[:, k - 1] = -3.0 * B[:, 0]
    if k > 3:
        B[:, 1] = 2.0 * B[:, 0]
    cg = pm.solvers.CG(preconditioner=pm.solvers.build_hierarchy(d, 2, omega=0.4, smooth_steps=2), tol=1e-10,
                       maxit=300)
    cg.update(K)
    X = cg.solve(B)
    assert cg.iterations < 300 and true_residual(K, X, B) < 2e-10
    assert float((X[:, k - 1] + 3.0 * X[:, 0]).abs().max() / X.abs().max()) < 1e-7


@pytest.mark.parametrize("k", [2, 5])
def test_columns_through_every_level_operator(gpu_lib, k):
    """The same solve through each operator that takes several columns: level 1 stored or stencil-free, the fine
    grid's kernels (all columns in one launch or one each) and the matrix-core sweeps.  A wrong column would
    cost the preconditioner its effect: the iteration counts agree (two more with BF16 sweeps)."""
    from pymoto_amd import tune
    d, K, B = problem((24, 16, 8), k, 7)
    its = {}
    try:
        for free in (False, True):
            for kernel in (0, 1, 2):
                for prec in ("fp64", "fp32", "bf16"):
                    tune.set_coarse_level1(free)
                    tune.set_tuning(fine_kernel=kernel)
                    mg = pm.solvers.build_hierarchy(d, 3, omega=0.4, smooth_steps=2, precision=prec)
                    cg = pm.solvers.CG(preconditioner=mg, tol=1e-10, maxit=300)
                    cg.update(K)
                    X = cg.solve(B)
                    assert true_residual(K, X, B) < 2e-10
                    its[free, kernel, prec] = cg.iterations
    finally:
        tune.set_coarse_level1(None)
        tune.set_tuning(**tune.DEFAULT)
    base = its[False, 0, "fp64"]
    assert all(abs(n - base) <= (2 if key[2] == "bf16" else 1) for key, n in its.items()), its


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_fewer_columns_on_the_same_handle(gpu_lib, prec, graph):
    """Blocks of falling and rising width on one handle, among them every width that the kernels round up (3, 5, 6, 7)
    after a wider one: the columns of the earlier block leave nothing behind."""
    d, K, B = problem((12, 8, 4), 15, 11)
    mg = pm.solvers.build_hierarchy(d, 2, omega=0.4, smooth_steps=2, precision=prec)
    cg = pm.solvers.CG(preconditioner=mg, tol=1e-10, maxit=300, graph=graph)
    cg.update(K)
    for k in (4, 3, 2, 4, 3, 8, 5, 3, 7, 2, 6, 1, 5, 8):
        X = cg.solve(B[:, :k].contiguous())
        assert cg.iterations < 300 and true_residual(K, X, B[:, :k]) < 2e-10, k
    for k in (11, 13, 14, 15):  # one call, blocks of 8 and of 3, 5, 6 and 7 columns
        X = cg.solve(B[:, :k].contiguous())
        assert cg.iterations < 300 and true_residual(K, X, B[:, :k]) < 2e-10, k


def test_solved_columns_leave_the_block(gpu_lib):
    """Four loads, then four of which one is known: the linear dependency aware solver passes on three."""
    d, K, B = problem((12, 8, 4), 8, 12)
    mg = pm.solvers.build_hierarchy(d, 2, omega=0.4, smooth_steps=2)
    lda = pm.solvers.LDAWrapper(pm.solvers.CG(preconditioner=mg, tol=1e-10, maxit=300), tol=1e-9)
    lda.update(K)
    lda.solve(B[:, :4].contiguous())
    B[:, 5] = B[:, 0] - 2.0 * B[:, 3]
    X = lda.solve(B[:, 4:].contiguous())
    assert true_residual(K, X, B[:, 4:]) < 2e-9
