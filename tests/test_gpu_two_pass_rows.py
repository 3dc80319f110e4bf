"""The two-pass coherent sum and its adjoint on the row-major column fields, at
every coarse size of the table (144 to 1024: groups of 10 to 32 lanes), windows of few and many columns, odd and even, on and off the centre,
single kernels and several groups of them, against float64 transforms.

Tolerances as for the other image transforms of these lengths: 6e-6 of the peak
pixel, 1.2e-5 of the peak gradient."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import engine
from test_gpu_dft_sizes import GRAD_TOL, IMAGE_TOL, _gradient, _image, _kernels

pytestmark = pytest.mark.gpu

# ny, nx, window rows (k0r, wr), window columns (k0c, wc), kernels, batch, coarse size
SIZES = [
    (256, 320, (-34, 70), (-33, 67), 3, 2, 144),
    (320, 256, (-30, 71), (-3, 5), 1, 1, 144),       # five columns: one part-filled block
    (512, 512, (-55, 111), (-55, 111), 12, 3, 256),
    (288, 512, (-64, 128), (-40, 65), 2, 1, 256),    # the widest window of 256
    (256, 320, (-50, 100), (-36, 73), 4, 2, 200),
    (640, 512, (-60, 131), (-9, 17), 5, 1, 324),
    (512, 640, (-100, 200), (-81, 163), 2, 2, 400),
    (512, 640, (-112, 225), (-107, 215), 3, 2, 450),
    (576, 576, (-128, 256), (-120, 231), 2, 1, 512),
    (1024, 640, (-140, 288), (-144, 270), 2, 3, 576),
    (1024, 960, (-200, 401), (-30, 61), 2, 1, 900),
    (1080, 2048, (-250, 500), (-256, 512), 1, 2, 1024),
]


@pytest.mark.parametrize("ny,nx,rows,cols,K,batch,coarse", SIZES)
def test_image_and_gradient(gpu, ny, nx, rows, cols, K, batch, coarse):
    ks, full = _kernels(ny, nx, rows, cols, K, ny + K)
    plan = engine.plan_for(ks, 1, batch)
    assert (plan.info()["path"], plan.info()["lr"]) == (2, coarse)
    rng = np.random.default_rng(nx)
    h = rng.random((batch, ny, nx)).astype(np.float32)
    g = rng.standard_normal((batch, ny, nx)).astype(np.float32)
    hd, gd = torch.as_tensor(h).cuda(), torch.as_tensor(g).cuda()
    img = engine.socs_image(hd, ks, pack_real=False).cpu().numpy()
    grad = engine.socs_adjoint(hd, gd, ks, pack_real=False).cpu().numpy()
    for b in range(batch):
        ref = _image(full, h[b])
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()
        ref = _gradient(full, h[b], g[b])
        assert np.max(np.abs(grad[b] - ref)) <= GRAD_TOL * np.abs(ref).max()


# the one-pass path's grids of 100 and 128, summed in two passes: window, channels, kernels, batch
SPLIT = [
    (128, 192, (-24, 48), (-25, 50), 1, 7, 3, 100),
    (192, 128, (-2, 4), (-20, 45), 3, 1, 1, 100),
    (256, 256, (-31, 64), (-28, 57), 3, 24, 2, 128),
    (160, 512, (-30, 61), (-40, 52), 2, 3, 4, 128),
]


@pytest.mark.parametrize("ny,nx,rows,cols,nchan,K,batch,coarse", SPLIT)
def test_split_sum_of_fields(gpu, ny, nx, rows, cols, nchan, K, batch, coarse):
    from opticalimaging_amd import _native as nat
    ks, full = _kernels(ny, nx, rows, cols, K, ny + K)
    plan = engine.plan_for(ks, nchan, batch)
    assert plan.info()["path"] < 2 and plan.info()["lr"] == coarse
    rng = np.random.default_rng(nx)
    f = (rng.standard_normal((batch, ny, nx, 3)) + 1j * rng.standard_normal((batch, ny, nx, 3))).astype(np.complex64)
    chans = [2, 0, 1][:nchan]
    img = engine.socs_image(torch.as_tensor(f).cuda(), ks, kind=nat.OI_FIELD_C64_CHLAST, cin=3,
                            chans=chans).cpu().numpy()
    for b in range(batch):
        ref = sum(_image(full, f[b, :, :, c]) for c in chans)
        assert np.max(np.abs(img[b] - ref)) <= IMAGE_TOL * ref.max()
    if nchan == 1:
        h, g = rng.random((2, batch, ny, nx)).astype(np.float32)
        out = engine.socs_adjoint(torch.as_tensor(h).cuda(), torch.as_tensor(g).cuda(), ks,
                                  pack_real=False).cpu().numpy()
        for b in range(batch):
            ref = _gradient(full, h[b], g[b])
            assert np.max(np.abs(out[b] - ref)) <= GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("K,batch", [(1700, 6), (2300, 2)])
def test_split_sum_beyond_its_bounds(gpu, K, batch):
    """Column fields of 104 MB an image (chunks of five images) and of 141 MB
    (the one-pass kernel) against one kernel set split over two calls: the same
    squares in another order, K 2^-24 of the peak."""
    g = torch.Generator(device="cuda").manual_seed(K)
    win = torch.randn((K, 60, 60), dtype=torch.complex64, device="cuda", generator=g)
    m = torch.rand((batch, 192, 160), device="cuda", generator=g)
    def image(w):
        ks = engine.KernelSet(w.contiguous(), -30, -30, 192, 160)
        return engine.socs_image(m, ks, pack_real=False)
    out = image(win)
    ref = image(win[:K // 2]) + image(win[K // 2:])
    assert (out - ref).abs().max() <= K * 2.0 ** -24 * ref.max()
