"""The Q4 V-cycle whose sweeps of a level run in one launch, against the oracle's V-cycle: sweep counts from the
smallest to the largest that a block's halo allows (10) and one beyond (the launches per sweep), grids with fewer
nodes than a block and with ragged last blocks, Dirichlet dofs on a face, in the interior and on single
components, damped Jacobi and Chebyshev.

Tolerances: FP64 1e-9 of the result's largest entry, as the other V-cycle tests (the oracle factorises the
coarsest matrix, the device inverts it); FP32 1e-4: some hundred operations at 6e-8 each, amplified by the
coarsest solve."""
import numpy as np
import pytest
import torch

import pymoto_amd as pm
from oracle import fe
from oracle.solvers import GeometricMultigrid as OGMG
from oracle.solvers import build_mg

pytestmark = pytest.mark.gpu

GRIDS = [((8, 4), 2), ((12, 10), 2), ((64, 4), 2), ((36, 20), 3), ((120, 40), 4), ((52, 84), 3), ((130, 66), 2)]


def dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64).cuda()


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def problem(nel, seed):
    nx, ny = nel[0] + 1, nel[1] + 1
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.3, 1.0, nel[0] * nel[1])
    node = lambda i, j: j * nx + i
    bc = np.unique([2 * node(0, j) for j in range(ny)] + [2 * node(i, 0) + 1 for i in range(0, nx, 3)]
                   + [2 * node(nx // 2, ny // 2), 2 * node(nx // 2, ny // 2) + 1, 2 * node(nx - 1, ny - 1) + 1])
    return x, bc, rng.standard_normal(2 * nx * ny)


@pytest.mark.parametrize("steps", [1, 2, 5, 10, 11])
@pytest.mark.parametrize("nel,levels", GRIDS)
def test_q4_vcycle_vs_oracle(gpu_lib, nel, levels, steps):
    x, bc, r = problem(nel, steps)
    Kref = fe.Assembly(*nel, 0, fe.element_stiffness(2), bc=bc).matrix(x)
    omg = build_mg((*nel, 0), levels, omega=0.4, smooth_steps=steps)
    omg.update(Kref)
    d = pm.VoxelDomain(*nel)
    K = pm.AssembleStiffness(d, bc=bc)(dev(x))
    ref = omg.solve(r)
    for prec, tol in (("fp64", 1e-9), ("fp32", 1e-4)):
        mg = pm.solvers.build_hierarchy(d, levels, omega=0.4, smooth_steps=steps, precision=prec)
        mg.update(K)
        for _ in range(2):
            assert relerr(mg.solve(dev(r)).cpu().numpy(), ref) < tol, prec


class Cheb:
    """The device's Chebyshev smoother on the oracle's operator, with the device's interval."""

    def __init__(self, lo, hi, steps):
        self.t, self.d, self.n = 0.5 * (hi + lo), 0.5 * (hi - lo), steps

    def run(self, A, b, u):
        D = A.diagonal()
        s = self.t / self.d
        rho, prev, u = 1.0 / s, u, u + (b - A @ u) / D / self.t
        for _ in range(1, self.n):
            new = 1.0 / (2.0 * s - rho)
            u, prev = u + 2.0 * new / self.d * (b - A @ u) / D + new * rho * (u - prev), u
            rho = new
        return u


def cheb_cycle(lvl, cheb, b):
    u = cheb[0].run(lvl.A, b, np.zeros_like(b))
    rc = lvl.R.T @ (b - lvl.A @ u)
    e = cheb_cycle(lvl.inner, cheb[1:], rc) if isinstance(lvl.inner, OGMG) else lvl.inner.solve(rc)
    return cheb[0].run(lvl.A, b, u + lvl.R @ e)


@pytest.mark.parametrize("steps", [1, 3, 10])
@pytest.mark.parametrize("nel,levels", [((36, 20), 3), ((130, 66), 2)])
def test_q4_chebyshev_vcycle_vs_oracle(gpu_lib, nel, levels, steps):
    x, bc, r = problem(nel, steps)
    Kref = fe.Assembly(*nel, 0, fe.element_stiffness(2), bc=bc).matrix(x)
    omg = build_mg((*nel, 0), levels, omega=0.4, smooth_steps=steps)
    omg.update(Kref)
    d = pm.VoxelDomain(*nel)
    mg = pm.solvers.build_hierarchy(d, levels, omega="chebyshev", smooth_steps=steps)
    mg.update(pm.AssembleStiffness(d, bc=bc)(dev(x)))
    cheb = [Cheb(*mg.smoother_interval(l), steps) for l in range(levels - 1)]
    assert relerr(mg.solve(dev(r)).cpu().numpy(), cheb_cycle(omg, cheb, r)) < 1e-9


@pytest.mark.parametrize("steps", [1, 2, 8, 10])
def test_q4_large_level_by_launches(gpu_lib, steps):
    """A fine grid (164,000 nodes) above the size up to which a visit of 1, 8 and 10 sweeps goes in one launch, over levels
    below it; 2 sweeps still do.  The V-cycle, and CG with one and with three columns, whose update forms the first sweep."""
    nel, levels = (1024, 160), 4
    x, bc, r = problem(nel, steps)
    Kref = fe.Assembly(*nel, 0, fe.element_stiffness(2), bc=bc).matrix(x)
    omg = build_mg((*nel, 0), levels, omega=0.4, smooth_steps=steps)
    omg.update(Kref)
    d = pm.VoxelDomain(*nel)
    K = pm.AssembleStiffness(d, bc=bc)(dev(x))
    ref = omg.solve(r)
    B = torch.stack([dev(r), dev(np.roll(r, 2)), dev(r * r)], dim=1)
    B[torch.as_tensor(bc)] = 0.0
    its = {}
    for prec, tol in (("fp64", 1e-9), ("fp32", 1e-4)):
        mg = pm.solvers.build_hierarchy(d, levels, omega=0.4, smooth_steps=steps, precision=prec)
        cg = pm.solvers.CG(preconditioner=mg, tol=1e-8, maxit=1000)
        cg.update(K)
        assert relerr(mg.solve(dev(r)).cpu().numpy(), ref) < tol, prec
        for b in (B[:, 0].contiguous(), B):
            u = cg.solve(b)
            its[prec, b.ndim] = cg.iterations
            assert cg.iterations < 1000 and float((K.residual(B[:, 0].contiguous(), u if u.ndim == 1 else u[:, 0].contiguous())
                                                  ).norm() / B[:, 0].norm()) < 2e-8, prec
    assert abs(its["fp64", 1] - its["fp32", 1]) <= 2 and abs(its["fp64", 2] - its["fp32", 2]) <= 2, its
