"""The convolution kernels of the warm-start network at the edges of their boxes: every channel pair on grids
that the boxes of output voxels do and do not divide, down to one box, against 64-bit sums.

Tolerances from the arithmetic: a sum of n products in FP32, whatever the order, is off by at most
n 2^-24 sum|a b|; a BF16 result adds half an ulp, 2^-9 |y| (and the ReLU adds nothing)."""
import numpy as np
import pytest
import torch

from pymoto_amd import _lib

pytestmark = pytest.mark.gpu

PAIRS = [(8, 16), (16, 16), (16, 32), (16, 64), (32, 16), (32, 32), (32, 64), (64, 16), (64, 32), (64, 64)]
GRIDS = [(4, 4, 4), (16, 1, 1), (1, 1, 16), (2, 8, 3), (12, 20, 5), (33, 16, 3), (40, 12, 9)]


def windows(t, shape):
    tp = torch.nn.functional.pad(t.reshape(*shape, -1), (0, 0, 1, 1, 1, 1, 1, 1))
    return [tp[tuple(slice(a, a + m) for a, m in zip((k // 9, (k // 3) % 3, k % 3), shape))].reshape(-1, t.shape[-1])
            for k in range(27)]


def run(nel, ci, co, X, W, b, dY, relu):
    lib, p, st = _lib.lib(), _lib.ptr, _lib.stream()
    n = X.shape[0]
    Y = torch.full((n + 16, co), 7.0, dtype=torch.bfloat16, device="cuda")  # 16 rows behind the result stay as they are
    dW = torch.empty(27, co, ci, dtype=torch.float32, device="cuda")
    db = torch.empty(co, dtype=torch.float32, device="cuda")
    work = torch.full((lib.pmt_conv3d_wgrad_work_size(ci, co),), float("nan"), dtype=torch.float32, device="cuda")
    _lib.check(lib.pmt_conv3d_fwd(*nel, ci, co, p(X), p(W), p(b), relu, p(Y), st))
    _lib.check(lib.pmt_conv3d_bwd_weight(*nel, ci, co, p(X), p(dY), p(dW), p(db), p(work), st))
    dX = None
    if ci >= 16:
        dX = torch.empty(n, ci, dtype=torch.bfloat16, device="cuda")
        Wt = torch.empty_like(W)
        _lib.check(lib.pmt_conv3d_bwd_data(*nel, ci, co, p(dY), p(W), p(Wt), p(dX), st))
    assert bool((Y[n:] == 7.0).all())
    return Y[:n], dW, db, dX


def close(got, ref, bound):
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound.clamp_min(1e-300)).max())


@pytest.mark.parametrize("ci,co", PAIRS)
@pytest.mark.parametrize("nel", GRIDS)
def test_conv_boxes(gpu_lib, ci, co, nel):
    n = int(np.prod(nel))
    g = torch.Generator().manual_seed(n * 1000 + ci * 64 + co)
    X = torch.randn(n, ci, generator=g).to(torch.bfloat16).cuda()
    W = (torch.randn(27, co, ci, generator=g) * 0.1).to(torch.bfloat16).cuda()
    b = torch.randn(co, generator=g).cuda()
    dY = torch.randn(n, co, generator=g).to(torch.bfloat16).cuda()
    if n % 16:
        with pytest.raises(_lib.HIPError):
            run(nel, ci, co, X, W, b, dY, 1)
        return
    Y, dW, db, dX = run(nel, ci, co, X, W, b, dY, 1)
    shape = tuple(reversed(nel))
    Xw, Gw = windows(X.double(), shape), windows(dY.double(), shape)
    Wd, Gd = W.double(), dY.double()
    u = 2.0 ** -24
    y = b.double() + sum(Xw[t] @ Wd[t].T for t in range(27))
    ya = b.double().abs() + sum(Xw[t].abs() @ Wd[t].abs().T for t in range(27))
    close(Y, y.clamp_min(0.0), 2.0 ** -8 * y.abs() + 27 * ci * u * ya)
    dw = torch.stack([Gd.T @ Xw[t] for t in range(27)])
    dwa = torch.stack([Gd.abs().T @ Xw[t].abs() for t in range(27)])
    close(dW, dw, n * u * dwa + 1e-30)
    close(db, Gd.sum(0), n * u * Gd.abs().sum(0) + 1e-30)
    if dX is not None:
        dx = sum(Gw[26 - t] @ Wd[t] for t in range(27))
        dxa = sum(Gw[26 - t].abs() @ Wd[t].abs() for t in range(27))
        close(dX, dx, 2.0 ** -8 * dx.abs() + 27 * co * u * dxa)


@pytest.mark.parametrize("ci,co", [(8, 16), (16, 16), (64, 64)])
@pytest.mark.parametrize("nel", [(12, 20, 5), (16, 8, 8)])
def test_conv_non_finite_voxel_stays_local(gpu_lib, ci, co, nel):
    """An infinite activation on the far corner reaches exactly the outputs and weight offsets that use it."""
    n = int(np.prod(nel))
    g = torch.Generator().manual_seed(5)
    X = torch.randn(n, ci, generator=g).to(torch.bfloat16)
    X[n - 1, 0] = float("inf")  # voxel (nx - 1, ny - 1, nz - 1), channel 0
    W = (torch.randn(27, co, ci, generator=g) * 0.1).to(torch.bfloat16)
    b = torch.zeros(co)
    dY = (torch.rand(n, co, generator=g) + 0.5).to(torch.bfloat16)
    Y, dW, db, _ = run(nel, ci, co, X.cuda(), W.cuda(), b.cuda(), dY.cuda(), 0)
    shape = tuple(reversed(nel))
    hit = torch.zeros(shape, dtype=torch.bool)
    hit[-2:, -2:, -2:] = True
    assert torch.equal(~torch.isfinite(Y.float()).cpu(), hit.reshape(-1, 1).expand(-1, co))
    # offset (dx, dy, dz) reads the corner from the voxel at corner - offset: inside the grid for offsets >= 0
    bad = ~torch.isfinite(dW).cpu()
    want = torch.zeros_like(bad)
    for t in range(27):
        if t // 9 >= 1 and (t // 3) % 3 >= 1 and t % 3 >= 1:
            want[t, :, 0] = True
    assert torch.equal(bad, want)
    assert bool(torch.isfinite(db).all())


@pytest.mark.parametrize("ci,co", [(8, 16), (16, 16), (32, 64), (64, 64)])
@pytest.mark.parametrize("nel", [(56, 20, 8), (40, 12, 12), (88, 16, 8)])
def test_conv_non_finite_voxel_beside_an_outer_group(gpu_lib, ci, co, nel):
    """The same where whole groups of 8 voxels of the last box lie outside the grid."""
    test_conv_non_finite_voxel_stays_local(gpu_lib, ci, co, nel)
