"""Windows much wider than a kernel's band: past the smallest coarse grid of the
band (the next one that holds the window serves), and too wide for the LDS tile of
the register row transform (nx = 1024: 692 columns, nx = 512: 356).  Image and
gradient against float64.  Tolerances as for the other image transforms of these
lengths."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import engine
from test_gpu_dft_sizes import GRAD_TOL, IMAGE_TOL, _gradient, _image

pytestmark = pytest.mark.gpu


def _set(ny, nx, wr, wc, bc, K):
    """Kernels of bc columns anywhere in the window, and their full spectra."""
    rng = np.random.default_rng(wc)
    win = np.zeros((K, wr, wc), np.complex64)
    for k in range(K):
        j = (wc - bc) * k // max(1, K - 1)
        win[k, :, j:j + bc] = (rng.standard_normal((wr, bc)) + 1j * rng.standard_normal((wr, bc))) / 8
    full = np.zeros((K, ny, nx), np.complex128)
    full[np.ix_(range(K), (np.arange(wr) - wr // 2) % ny, (np.arange(wc) - wc // 2) % nx)] = win
    return engine.KernelSet(torch.as_tensor(win).cuda(), -(wr // 2), -(wc // 2), ny, nx, band=(wr, bc)), full


@pytest.mark.parametrize("ny,nx,wr,wc,bc", [(1024, 1024, 30, 800, 440), (1024, 1024, 30, 692, 440),
                                            (512, 512, 21, 380, 190), (512, 512, 21, 356, 190)])
def test_image(gpu, ny, nx, wr, wc, bc):
    ks, full = _set(ny, nx, wr, wc, bc, 3)
    h = np.random.default_rng(ny).random((2, ny, nx)).astype(np.float32)
    img = engine.socs_image(torch.as_tensor(h).cuda(), ks, pack_real=False).cpu().numpy()
    for b in range(2):
        ref = _image(full, h[b])
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()


@pytest.mark.parametrize("ny,nx,wr,wc,bc,coarse", [(512, 512, 30, 234, 90, 256), (648, 540, 31, 330, 95, 400),
                                                   (1024, 640, 33, 401, 150, 450), (2048, 1024, 9, 577, 110, 900)])
def test_coarse_grid_of_the_window(gpu, ny, nx, wr, wc, bc, coarse):
    ks, full = _set(ny, nx, wr, wc, bc, 3)
    info = engine.plan_for(ks, 1, 1).info()
    assert (info["path"], info["lr"]) == (2, coarse)
    h, g = np.random.default_rng(wc).random((2, ny, nx)).astype(np.float32)
    hd, gd = torch.as_tensor(h[None]).cuda(), torch.as_tensor(g[None]).cuda()
    ref = _image(full, h)
    assert np.max(np.abs(engine.socs_image(hd, ks, pack_real=False).cpu().numpy()[0] - ref)) <= IMAGE_TOL * ref.max()
    ref = _gradient(full, h, g)
    out = engine.socs_adjoint(hd, gd, ks, pack_real=False).cpu().numpy()[0]
    assert np.max(np.abs(out - ref)) <= GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("ny,nx,wr,wc,bc", [(512, 512, 21, 190, 190), (1024, 1024, 30, 800, 440)])
def test_gradient(gpu, ny, nx, wr, wc, bc):
    """The image's own band, twice a kernel's, is what the cotangent's rows keep."""
    ks, full = _set(ny, nx, wr, wc, bc, 3)
    h, g = np.random.default_rng(nx).standard_normal((2, 2, ny, nx)).astype(np.float32)
    out = engine.socs_adjoint(torch.as_tensor(h).cuda(), torch.as_tensor(g).cuda(), ks, pack_real=False).cpu().numpy()
    for b in range(2):
        ref = _gradient(full, h[b], g[b])
        assert np.max(np.abs(out[b] - ref)) <= GRAD_TOL * np.abs(ref).max()


def test_optimisation_steps(gpu):
    """Refused by the band form and taken by the general one."""
    from opticalimaging_amd import ILT
    ks, _ = _set(512, 512, 21, 380, 190, 2)
    gen = torch.Generator(device="cuda").manual_seed(1)
    target = (torch.rand((1, 512, 512), device="cuda", generator=gen) < 0.4).float()
    theta = torch.randn((1, 512, 512), device="cuda", generator=gen)
    out = ILT.ilt(theta, target, ks, steps=2)
    assert all(torch.isfinite(x).all() for x in out if isinstance(x, torch.Tensor))
