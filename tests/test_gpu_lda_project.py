"""The device-side projection of the linear dependency aware solver, r -= a b and y += sign a x with
a = (r . b) / (b . b), against torch in FP64: below one block, at and around a block's 1,024 entries, and more entries
than the partial sums' blocks take at once.  Tolerance: a is a quotient of sums of n terms, 1e-12 relative; the updates
add two roundings."""
import pytest
import torch

import pymoto_amd as pm  # noqa: F401
from pymoto_amd.solvers.solvers import _project

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 70001, 300001])
@pytest.mark.parametrize("sign", [1.0, -1.0, None])
def test_projection(gpu_lib, n, sign):
    g = torch.Generator().manual_seed(n)
    b, x, r, y = (torch.randn(n, generator=g, dtype=torch.float64).cuda() for _ in range(4))
    a = float(r.dot(b) / b.dot(b))
    r_ref, y_ref = r - a * b, y + (sign or 0.0) * a * x
    if sign is None:
        _project(b, r)
    else:
        _project(b, r, x, y, sign)
    scale = float(r.dot(r).sqrt() / b.dot(b).sqrt()) + abs(a)
    assert float((r - r_ref).abs().max()) <= 1e-12 * scale * float(b.abs().max()) + 1e-15 * float(r_ref.abs().max())
    assert float((y - y_ref).abs().max()) <= 1e-12 * scale * float(x.abs().max()) + 1e-15 * float(y_ref.abs().max())
