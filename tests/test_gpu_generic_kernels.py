"""The kernels for any length, which a coarse grid of the caller's choice selects
(plans of every other geometry run compile-time sizes or matrix products): images of
real masks and of complex fields, and the mask gradient, against float64.
Tolerances as for the other transforms of these lengths."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import _native as nat
from opticalimaging_amd import engine
from test_gpu_dft_sizes import GRAD_TOL, IMAGE_TOL, _gradient, _image, _kernels

pytestmark = pytest.mark.gpu

# grid, window rows, window columns, kernels, batch, coarse grid
SIZES = [((96, 160), (-9, 19), (-10, 21), 5, 3, (40, 48)), ((60, 90), (-6, 12), (-8, 17), 3, 2, (24, 36)),
         ((128, 256), (-12, 25), (-20, 40), 4, 2, (50, 80)), ((135, 405), (-15, 31), (-30, 61), 2, 1, (64, 125)),
         ((512, 300), (-50, 101), (-40, 81), 2, 2, (216, 162))]


def _plan(grid, rows, cols, K, batch, coarse, nchan=1):
    plan = engine.Plan(*grid, *rows, *cols, nchan=nchan, max_batch=batch, lr=coarse[0], lc=coarse[1], max_kernels=K)
    i = plan.info()
    assert (i["path"], i["direct"], i["lr"], i["lc"]) == (0, 0, *coarse)
    return plan


@pytest.mark.parametrize("grid,rows,cols,K,batch,coarse", SIZES)
def test_masks(gpu, grid, rows, cols, K, batch, coarse):
    ks, full = _kernels(*grid, rows, cols, K, K)
    plan = _plan(grid, rows, cols, K, batch, coarse)
    rng = np.random.default_rng(grid[1])
    h, g = rng.random((batch, *grid)).astype(np.float32), rng.standard_normal((batch, *grid)).astype(np.float32)
    hd, gd = torch.as_tensor(h).cuda(), torch.as_tensor(g).cuda()
    img = engine.socs_image(hd, ks, plan=plan, pack_real=False).cpu().numpy()
    grad = engine.socs_adjoint(hd, gd, ks, plan=plan, pack_real=False).cpu().numpy()
    for b in range(batch):
        ref = _image(full, h[b])
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()
        ref = _gradient(full, h[b], g[b])
        assert np.max(np.abs(grad[b] - ref)) <= GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("grid,rows,cols,K,batch,coarse", SIZES)
def test_fields(gpu, grid, rows, cols, K, batch, coarse):
    ks, full = _kernels(*grid, rows, cols, K, K)
    plan = _plan(grid, rows, cols, K, batch, coarse, 2)
    rng = np.random.default_rng(grid[0])
    f = (rng.standard_normal((batch, *grid, 3)) + 1j * rng.standard_normal((batch, *grid, 3))).astype(np.complex64)
    img = engine.socs_image(torch.as_tensor(f).cuda(), ks, kind=nat.OI_FIELD_C64_CHLAST, cin=3, chans=[2, 0],
                            plan=plan).cpu().numpy()
    for b in range(batch):
        ref = _image(full, f[b, :, :, 2]) + _image(full, f[b, :, :, 0])
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()
