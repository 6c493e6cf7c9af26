"""The wide FilterConv kernels (radii above 3, extents that are not equal on all axes) against the per-element
gather kernels: the taps are summed in the same order, so forward and adjoint have the same bits for every face
condition, at the edges of the boxes (32 x 8 x 4 outputs, 32 x 32 in 2D) and with elements that meet two faces."""
import numpy as np
import numpy.testing as npt
import pytest
import torch

import pymoto_amd as pm
from oracle.filter import ConvFilter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,radius", [((32, 8, 4), 3.4), ((33, 9, 5), 3.4), ((70, 17, 13), 4.6), ((7, 6, 11), 3.9),
                                        ((40, 21, 2), 3.4), ((19, 9, 1), 1.5), ((64, 32, 0), 3.4), ((65, 33, 0), 8.0),
                                        ((45, 70, 0), 5.2), ((13, 12, 12), 5.5)])
@pytest.mark.parametrize("bcs", [("symmetric",) * 6, ("edge", "wrap", "symmetric", 0.25, "wrap", "edge"),
                                 ("wrap",) * 6, (0.5, "edge", "wrap", "symmetric", "edge", 0.0)])
def test_filter_wide_equals_gather(gpu_lib, nel, radius, bcs):
    d = pm.VoxelDomain(*nel)
    kw = dict(zip(("xmin_bc", "xmax_bc", "ymin_bc", "ymax_bc", "zmin_bc", "zmax_bc"), bcs))
    rng = np.random.default_rng(int(radius * 10) + nel[0])
    x, dy = rng.uniform(0.0, 1.0, d.nel), rng.standard_normal(d.nel)
    out = {}
    try:
        for tiled in (1, 0):
            assert gpu_lib.pmt_set_tuning(6, tiled) == 0
            m = pm.FilterConv(d, radius=radius, **kw)
            sx = pm.Signal("x", torch.as_tensor(x).cuda())
            sy = m(sx)
            sy.sensitivity = torch.as_tensor(dy).cuda()
            m.sensitivity()
            out[tiled] = (sy.state.cpu().numpy(), sx.sensitivity.cpu().numpy())
    finally:
        gpu_lib.pmt_set_tuning(6, 1)
    npt.assert_array_equal(out[1][0], out[0][0])
    npt.assert_array_equal(out[1][1], out[0][1])
    filt = ConvFilter(nel, m.weights, (bcs[0:2], bcs[2:4], bcs[4:6]))
    npt.assert_allclose(out[1][0], filt.forward(x), rtol=1e-12, atol=1e-14)
    npt.assert_allclose(out[1][1], filt.adjoint(dy), rtol=1e-12, atol=1e-13)


@pytest.mark.parametrize("shape", [(3, 3, 17), (3, 3, 19), (3, 3, 21), (3, 3, 35), (3, 3, 37), (5, 5, 9), (15, 15, 1), (7, 7, 3),
                                   (3, 5, 3)])
@pytest.mark.parametrize("nel", [(9, 7, 40), (200, 130, 70)])
def test_filter_unequal_extents(gpu_lib, shape, nel):
    """Weights that are not the same in z, up to the extents whose box just fits into LDS and the first that do not, with 2
    and with 4 outputs per thread: the bits of the gather kernels, with every kind of face in z."""
    d = pm.VoxelDomain(*nel)
    rng = np.random.default_rng(shape[2])
    w = rng.uniform(-1.0, 1.0, shape)
    x, dy = rng.uniform(0.0, 1.0, d.nel), rng.standard_normal(d.nel)
    out = {}
    try:
        for tiled in (1, 0):
            assert gpu_lib.pmt_set_tuning(6, tiled) == 0
            m = pm.FilterConv(d, weights=w, zmin_bc="wrap", zmax_bc=0.5, ymin_bc="edge")
            sx = pm.Signal("x", torch.as_tensor(x).cuda())
            sy = m(sx)
            sy.sensitivity = torch.as_tensor(dy).cuda()
            m.sensitivity()
            out[tiled] = (sy.state.cpu().numpy(), sx.sensitivity.cpu().numpy())
    finally:
        gpu_lib.pmt_set_tuning(6, 1)
    npt.assert_array_equal(out[1][0], out[0][0])
    npt.assert_array_equal(out[1][1], out[0][1])
    if nel[0] < 100:
        filt = ConvFilter(nel, w, (("symmetric",) * 2, ("edge", "symmetric"), ("wrap", 0.5)))
        npt.assert_allclose(out[1][0], filt.forward(x), rtol=1e-12, atol=1e-12)
        npt.assert_allclose(out[1][1], filt.adjoint(dy), rtol=1e-12, atol=1e-12)
