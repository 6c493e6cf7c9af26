"""The streamed hex8 sensitivity contraction u_e^T K0 v_e against its definition in torch, FP64: element counts at and
around a block's 15 x 15 columns, one layer up to more layers than one block walks, one and several terms, u the
same as v and not, and no term at all.  Tolerance: 24 x 24 products and transforms of 24 terms per element in FP64,
1e-12 of the largest entry."""
import numpy as np
import pytest
import torch

import pymoto_amd as pm
from oracle import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel", [(1, 1, 1), (15, 15, 1), (16, 14, 2), (14, 16, 3), (31, 30, 7), (45, 46, 40)])
@pytest.mark.parametrize("terms", [0, 1, 3])
def test_streamed_sensitivity(gpu_lib, nel, terms):
    d = pm.VoxelDomain(*nel)
    bc = problems.cantilever3d(*nel)[0]
    g = torch.Generator().manual_seed(nel[0] + terms)
    x = torch.rand(d.nel, generator=g, dtype=torch.float64).cuda() + 0.1
    sx = pm.Signal("x", x)
    mod = pm.AssembleStiffness(d, bc=bc)
    sK = mod(sx)
    K = sK.state
    n = K.shape[0]
    vec = [torch.randn(n, generator=g, dtype=torch.float64).cuda() for _ in range(4)]
    pairs = [(vec[0], vec[1], 0.7), (vec[2], vec[2], -1.3), (vec[3], vec[0], 2.0)][:terms]
    dm = pm.DyadicMatrix()
    for u, v, fac in pairs:
        dm.add_dyad(u, v, fac)
    got = mod._sensitivity(dm)
    K0 = K.grid.K0_dev[:576].reshape(24, 24)
    conn = torch.as_tensor(np.asarray(d.conn, dtype=np.int64)).cuda()
    dofs = (3 * conn[:, :, None] + torch.arange(3, device="cuda")).reshape(d.nel, 24)
    want = torch.zeros(d.nel, dtype=torch.float64, device="cuda")
    free = torch.ones(n, dtype=torch.float64, device="cuda")
    free[torch.as_tensor(np.asarray(bc, dtype=np.int64)).cuda()] = 0.0
    for u, v, fac in pairs:
        want += fac * (((free * u)[dofs] @ K0) * (free * v)[dofs]).sum(1)
    if not terms:
        assert float(got.abs().max()) == 0.0
    else:
        assert float((got.reshape(-1) - want).abs().max() / want.abs().max()) < 1e-12
