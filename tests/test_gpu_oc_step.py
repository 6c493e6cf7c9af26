"""The device-side OC bisection (pmt_oc_step) against the same bisection driven step by step with
pmt_oc_update: the same decisions and the same design, bit for bit, at the sizes where the multipliers per pass
and the number of blocks change, for designs on and off their bounds, zero and positive sensitivities."""
import warnings

import numpy as np
import pytest
import torch

import pymoto_amd as pm
from oracle.optim import oc_step
from pymoto_amd import _lib

pytestmark = pytest.mark.gpu


def stepwise(lib, x, dg, xmin, xmax, move, target, l1, l2, tol):
    xnew, tot = torch.full_like(x, -1.0), torch.empty(1, dtype=torch.float64, device="cuda")
    while l2 - l1 > tol:
        lmid = 0.5 * (l1 + l2)
        _lib.check(lib.pmt_oc_update(x.numel(), _lib.ptr(x), _lib.ptr(dg), xmin, xmax, move, lmid, _lib.ptr(xnew),
                                     _lib.ptr(tot), _lib.ptr(_lib.reduce_work()), _lib.stream()))
        if float(tot.item()) - target > 0:
            l1 = lmid
        else:
            l2 = lmid
    return xnew, l1, l2


@pytest.mark.parametrize("n", [1, 63, 257, 4800, 32768, 32769, 262144, 262145, 600001])
@pytest.mark.parametrize("kind", ["plain", "bounds", "signs", "negative"])
def test_oc_step_equals_stepwise(gpu_lib, n, kind):
    g = torch.Generator().manual_seed(n)
    x = torch.rand(n, generator=g, dtype=torch.float64)
    dg = -torch.rand(n, generator=g, dtype=torch.float64) ** 4
    xmin, xmax, move = 0.0, 1.0, 0.2
    if kind == "bounds":
        xmin, move = 1e-3, 0.05
        x = x.round().clamp(xmin, 1.0)
    if kind == "signs":
        dg[::3] = 0.0
        dg[1::7] *= -1.0
    if kind == "negative":
        xmin = -0.5
        x = x - 0.5
    target = (0.4 if kind != "negative" else 0.1) * n
    x, dg = x.cuda(), dg.cuda()
    for l1, l2, tol in ((0.0, 1e5, 1e-4), (0.3, 0.9, 1e-9), (0.0, 1.0, 0.4)):
        ref, r1, r2 = stepwise(gpu_lib, x, dg, xmin, xmax, move, target, l1, l2, tol)
        xnew = torch.full_like(x, -2.0)
        work = torch.full((gpu_lib.pmt_oc_work_size(),), float("nan"), dtype=torch.float64, device="cuda")
        _lib.check(gpu_lib.pmt_oc_step(n, _lib.ptr(x), _lib.ptr(dg), xmin, xmax, move, l1, l2, tol, target, _lib.ptr(xnew),
                                       _lib.ptr(work), _lib.stream()))
        s = work[:4].tolist()
        assert (s[0], s[1]) == (r1, r2) and s[3] == float(dg.max())
        assert torch.equal(xnew, ref)


def test_oc_module_warns_and_matches_oracle(gpu_lib):
    rng = np.random.default_rng(3)
    x, dg = rng.uniform(0.1, 0.9, 5000), -rng.uniform(0.0, 1.0, 5000) ** 3
    oc = pm.OC(pm.Signal("x", torch.as_tensor(x).cuda()), None, None, move=0.2, verbosity=0)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        new = oc.step(None, torch.as_tensor(dg).cuda())
    np.testing.assert_allclose(new.cpu().numpy(), oc_step(x, dg, move=0.2), rtol=1e-12)
    dg[7] = 0.5
    with pytest.warns(UserWarning, match="negative sensitivities"):
        oc.step(None, torch.as_tensor(dg).cuda())
    dg[8] = np.nan  # the largest sensitivity is not a number: no warning, as max() has it
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        oc.step(None, torch.as_tensor(dg).cuda())


def test_oc_refuses_multipliers_that_are_not_positive(gpu_lib):
    """The trial design x sqrt(-dg / l) needs l > 0: an interval whose bisection comes to another multiplier is
    refused, at its first step, at a later one or where the halvings underflow, and no other."""
    x = torch.full((100,), 0.5, dtype=torch.float64, device="cuda")
    dg = -torch.linspace(0.1, 1.0, 100, dtype=torch.float64, device="cuda")

    def step(l1, l2, tol, maxvol=0.5, d=dg):
        return pm.OC(pm.Signal("x", x), None, None, verbosity=0, l1init=l1, l2init=l2, l1l2tol=tol, maxvol=maxvol
                     ).step(None, d)

    for l1, l2, tol in ((-1.0, 1.0, 1e-4), (-3.0, 1.0, 1e-4), (float("-inf"), 1.0, 1e-4)):
        with pytest.raises(_lib.HIPError):  # first multiplier 0, -1, -inf
            step(l1, l2, tol)
    with pytest.raises(_lib.HIPError):  # 49.5, then below: every volume is less than the whole
        step(-1.0, 100.0, 1e-4, maxvol=1.0)
    with pytest.raises(_lib.HIPError):  # (0, l2] halved to nothing
        step(0.0, 1.0, 0.0, maxvol=1.0)
    # a negative end that no multiplier of the bisection reaches: as step by step
    ref, _, _ = stepwise(gpu_lib, x, 50.0 * dg, 0.0, 1.0, 0.1, 0.5 * 100, -1.0, 100.0, 1e-4)
    assert torch.equal(step(-1.0, 100.0, 1e-4, d=50.0 * dg), ref)
    work = torch.empty(gpu_lib.pmt_oc_work_size(), dtype=torch.float64, device="cuda")
    for l1, l2 in ((-1.0, 1.0), (float("nan"), 1.0), (0.0, float("inf"))):
        assert gpu_lib.pmt_oc_step(100, _lib.ptr(x), _lib.ptr(dg), 0.0, 1.0, 0.1, l1, l2, 1e-4, 50.0, _lib.ptr(x.clone()),
                                   _lib.ptr(work), _lib.stream()) < 0
