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


# windows on both sides of where products give way to transforms: real rows, complex
# rows and columns, even and odd lengths, plans of many images and of one
@pytest.mark.parametrize("ny,nx,wr,wc,bc", [(960, 1000, 256, 600, 200), (960, 1000, 257, 601, 200),
                                            (600, 405, 256, 256, 120), (405, 600, 257, 257, 120),
                                            (729, 640, 256, 257, 120), (640, 729, 257, 256, 120)])
@pytest.mark.parametrize("real,most", [(True, 16), (False, 16), (True, 2)])
def test_products_and_transforms(gpu, ny, nx, wr, wc, bc, real, most):
    from opticalimaging_amd import _native as nat
    rng = np.random.default_rng(wc)
    f = rng.standard_normal((2, ny, nx, 2)).astype(np.float32)
    h = f[..., 0] if real else f[..., 0] + 1j * f[..., 1]
    plan = engine.Plan(ny, nx, -(wr // 2), wr, -(wc // 2), wc, max_batch=most, band_r=bc, band_c=bc, max_kernels=1)
    assert plan.info()["path"] == 2
    hd = torch.as_tensor(h if real else h[..., None]).cuda()
    chans, keep = nat.int_array([0])
    kind = nat.OI_FIELD_REAL if real else nat.OI_FIELD_C64_CHLAST

    def spectrum(x):
        out = torch.empty((len(x), wr, wc), dtype=torch.complex64, device="cuda")
        nat.check(nat.load().oi_spectrum_window(plan.handle, nat.ptr(x), kind, 1, chans, len(x), nat.ptr(out),
                                                nat.stream()))
        return out
    out = spectrum(hd)
    ref = np.fft.ifft2(h.astype(np.complex128))
    ref = ref[:, (np.arange(wr) - wr // 2) % ny][:, :, (np.arange(wc) - wc // 2) % nx]
    # two transforms of one to seven hundred terms: half the image's tolerance
    assert np.max(np.abs(out.cpu().numpy() - ref)) <= IMAGE_TOL / 2 * np.abs(ref).max()
    assert torch.equal(spectrum(hd[1:]), out[1:])          # whatever the call's batch


@pytest.mark.parametrize("ny,nx,q", [(600, 640, 127), (600, 640, 128), (405, 675, 79), (405, 675, 80),
                                     (512, 675, 128), (675, 512, 128), (1125, 600, 90)])
def test_band_products_and_transforms(gpu, ny, nx, q):
    """Bands on both sides of where the products of their columns give way to
    transforms, and the gradient's last stage with them."""
    rng = np.random.default_rng(q)
    w = 2 * q + 1
    win = np.zeros((2, w, w), np.complex64)
    win[:, :q + 1, :q + 1] = (rng.standard_normal((2, q + 1, q + 1)) + 1j * rng.standard_normal((2, q + 1, q + 1))) / 8
    full = np.zeros((2, ny, nx), np.complex128)
    full[np.ix_(range(2), (np.arange(w) - q) % ny, (np.arange(w) - q) % nx)] = win
    ks = engine.KernelSet(torch.as_tensor(win).cuda(), -q, -q, ny, nx, band=(q + 1, q + 1))
    assert engine.plan_for(ks, 1, 10).info()["path"] == 2
    h, g = rng.random((2, 10, ny, nx)).astype(np.float32)
    img = engine.socs_image(torch.as_tensor(h).cuda(), ks, pack_real=False).cpu().numpy()
    grad = engine.socs_adjoint(torch.as_tensor(h).cuda(), torch.as_tensor(g).cuda(), ks, pack_real=False).cpu().numpy()
    for b in (0, 9):
        ref = _image(full, h[b])
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()
        ref = _gradient(full, h[b], g[b])
        assert np.max(np.abs(grad[b] - ref)) <= GRAD_TOL * np.abs(ref).max()


def test_lines_past_the_transforms(gpu):
    """12000 points stay products at any window: no LDS holds their transform."""
    from opticalimaging_amd import _native as nat
    ny, nx, wc = 960, 12000, 300
    rng = np.random.default_rng(5)
    win = (rng.standard_normal((1, 9, wc)) + 1j * rng.standard_normal((1, 9, wc))).astype(np.complex64)
    full = np.zeros((1, ny, nx), np.complex128)
    full[np.ix_([0], (np.arange(9) - 4) % ny, (np.arange(wc) - 150) % nx)] = win
    ks = engine.KernelSet(torch.as_tensor(win).cuda(), -4, -150, ny, nx)
    info = engine.plan_for(ks, 1, 1).info()
    assert (info["path"], info["lr"]) == (2, 900)
    h = (rng.standard_normal((1, ny, nx)) + 1j * rng.standard_normal((1, ny, nx))).astype(np.complex64)
    img = engine.socs_image(torch.as_tensor(h[..., None]).cuda(), ks, kind=nat.OI_FIELD_C64_CHLAST).cpu().numpy()
    ref = _image(full, h[0])
    assert np.max(np.abs(img[0] - ref)) <= IMAGE_TOL * ref.max()
