"""The row-wise restriction against the transposed linear interpolation written per axis, at row lengths around a
wavefront's 20 (3D) and 30 (2D) coarse nodes.  Tolerance: sums of 27 terms with weights up to 1, 1e-14 of the
largest value that enters times 27."""
import numpy as np
import pytest
import torch

import pymoto_amd as pm  # noqa: F401
from pymoto_amd import _lib

pytestmark = pytest.mark.gpu


def restrict_axis(v, axis):
    v = np.moveaxis(v, axis, 0)
    out = v[::2].copy()
    out[:-1] += 0.5 * v[1::2]
    out[1:] += 0.5 * v[1::2]
    return np.moveaxis(out, 0, axis)


@pytest.mark.parametrize("nel", [(2, 2, 2), (38, 4, 2), (40, 2, 4), (42, 6, 2), (78, 2, 2), (80, 4, 6), (2, 2, 0), (58, 4, 0),
                                 (60, 6, 0), (62, 2, 0), (118, 8, 0), (120, 40, 0)])
def test_restriction(gpu_lib, nel):
    dim = 3 if nel[2] else 2
    shape = [n + 1 for n in nel[::-1] if n] + [dim]
    r = np.random.default_rng(nel[0]).standard_normal(shape)
    want = r
    for axis in range(dim):
        want = restrict_axis(want, axis)
    out = torch.empty(want.size, dtype=torch.float64, device="cuda")
    lib = _lib.lib()
    _lib.check(lib.pmt_restrict(*nel, _lib.ptr(torch.as_tensor(r.ravel()).cuda()), _lib.ptr(out), _lib.stream()))
    assert np.abs(out.cpu().numpy().reshape(want.shape) - want).max() < 27e-14 * np.abs(r).max()
