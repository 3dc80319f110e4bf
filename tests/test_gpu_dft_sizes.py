"""Image lengths without a register transform (matrix products, csrc/oi_dft.hip):
images, mask gradients and optimisation steps against float64 numpy transforms
of the same kernels, over odd, even and mixed lengths (one length in the
register table, the other not), windows off centre, one to three channels, few
and many rows, and more orders than one workgroup takes.

Tolerances: a pixel is the end of four transforms of at most 2048 terms, summed
in chunks (root-of-terms growth, below 50 float32 roundings of 6e-8), times two
for the square: 6e-6 of the peak; gradients pass through twice as many: 1.2e-5."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import _native as nat
from opticalimaging_amd import engine

pytestmark = pytest.mark.gpu

IMAGE_TOL, GRAD_TOL = 6e-6, 1.2e-5

# ny, nx, window rows (k0r, wr), window columns (k0c, wc), batch
SIZES = [
    (96, 100, (-9, 19), (-10, 21), 3),          # smallest tiles, even
    (135, 225, (-15, 31), (-16, 33), 2),        # odd lengths, 16 orders and the 17th
    (225, 135, (-16, 33), (-15, 31), 1),
    (128, 375, (-12, 25), (-23, 50), 2),        # register length x product length, off centre
    (375, 128, (-27, 50), (-12, 25), 2),
    (405, 512, (-7, 30), (-31, 63), 1),         # window shifted to positive orders
    (640, 288, (-55, 111), (-8, 17), 4),
    (72, 640, (-8, 17), (-15, 31), 120),        # many rows: 64-row tiles
    (600, 810, (-31, 63), (-43, 87), 24),
    (1125, 1200, (-55, 111), (-60, 121), 5),
    (720, 1920, (-40, 81), (-107, 215), 4),     # seven order tiles
]
IDS = ["%dx%d b%d" % (s[0], s[1], s[4]) for s in SIZES]


def _kernels(ny, nx, rows, cols, K, seed):
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((K, rows[1], cols[1], 2)).astype(np.float32)
    win = w[..., 0] + 1j * w[..., 1]
    ks = engine.KernelSet(torch.as_tensor(win).cuda(), rows[0], cols[0], ny, nx)
    full = np.zeros((K, ny, nx), dtype=np.complex128)
    r = (rows[0] + np.arange(rows[1])) % ny
    c = (cols[0] + np.arange(cols[1])) % nx
    full[:, r[:, None], c[None, :]] = win
    return ks, full


def _fields(full, h):
    return np.fft.fft2(full * np.fft.ifft2(h.astype(np.complex128)))


def _image(full, h):
    return (np.abs(_fields(full, h)) ** 2).sum(0)


def _gradient(full, h, g):
    """d/dh of sum g I: 2 Re sum_k conj-correlation of the fields."""
    a = np.fft.fft2(g * np.conj(_fields(full, h)))
    return 2 * np.fft.ifft2((full * a).sum(0)).real


@pytest.mark.parametrize("size", SIZES, ids=IDS)
def test_images_of_real_masks(gpu, size):
    ny, nx, rows, cols, B = size
    ks, full = _kernels(ny, nx, rows, cols, 3, 1)
    m = np.random.default_rng(2).random((B, ny, nx)).astype(np.float32)
    out = engine.socs_image(torch.as_tensor(m).cuda(), ks).cpu().numpy()
    for b in sorted({0, B // 2, B - 1}):
        ref = _image(full, m[b])
        assert np.max(np.abs(out[b] - ref)) < IMAGE_TOL * ref.max()


@pytest.mark.parametrize("chans", [[0], [1], [0, 2], [0, 1, 2]])
@pytest.mark.parametrize("size", SIZES[:6] + [SIZES[9]], ids=IDS[:6] + [IDS[9]])
def test_images_of_complex_fields(gpu, size, chans):
    ny, nx, rows, cols, B = size
    ks, full = _kernels(ny, nx, rows, cols, 2, 3)
    rng = np.random.default_rng(4)
    f = (rng.standard_normal((B, ny, nx, 3)) + 1j * rng.standard_normal((B, ny, nx, 3))).astype(np.complex64)
    out = engine.socs_image(torch.as_tensor(f).cuda(), ks, kind=nat.OI_FIELD_C64_CHLAST, cin=3,
                            chans=chans).cpu().numpy()
    for b in {0, B - 1}:
        ref = sum(_image(full, f[b, :, :, c]) for c in chans)
        assert np.max(np.abs(out[b] - ref)) < IMAGE_TOL * ref.max()


@pytest.mark.parametrize("size", SIZES, ids=IDS)
def test_mask_gradients(gpu, size):
    ny, nx, rows, cols, B = size
    ks, full = _kernels(ny, nx, rows, cols, 2, 5)
    rng = np.random.default_rng(6)
    m = rng.random((B, ny, nx)).astype(np.float32)
    g = rng.standard_normal((B, ny, nx)).astype(np.float32)
    out = engine.socs_adjoint(torch.as_tensor(m).cuda(), torch.as_tensor(g).cuda(), ks).cpu().numpy()
    for b in {0, B - 1}:
        ref = _gradient(full, m[b], g[b])
        assert np.max(np.abs(out[b] - ref)) < GRAD_TOL * np.abs(ref).max()


@pytest.mark.parametrize("size", SIZES, ids=IDS)
def test_optimisation_step(gpu, size):
    """ILT.ilt, which takes the image and residual passes at these lengths."""
    from opticalimaging_amd import ILT
    ny, nx, rows, cols, B = size
    ks, full = _kernels(ny, nx, rows, cols, 2, 7)
    full = full / np.sqrt(ny * nx)
    ks = engine.KernelSet(ks.win / np.sqrt(ny * nx), ks.k0r, ks.k0c, ny, nx)
    rng = np.random.default_rng(8)
    th = rng.standard_normal((B, ny, nx)).astype(np.float32)
    m = 1 / (1 + np.exp(-th.astype(np.float64)))
    T = (rng.random((B, ny, nx)) > 0.5).astype(np.float32)
    img = np.stack([_image(full, x) for x in m])
    loss = ((img - T) ** 2).sum()
    grad = np.stack([_gradient(full, x, 2 * (i - t)) for x, i, t in zip(m, img, T)])
    theta, losses = ILT.ilt(torch.as_tensor(th).cuda(), torch.as_tensor(T).cuda(), ks, steps=1, lr=0.5)
    assert abs(float(losses[0]) - loss) < 1e-5 * loss
    gt = grad * m * (1 - m)
    step = 0.5 * gt / np.sqrt((gt ** 2).mean((1, 2), keepdims=True))
    assert np.max(np.abs(theta.cpu().numpy() - (th - step))) < 2 * GRAD_TOL * np.abs(step).max()


def test_without_allocation(gpu):
    """oi_socs_image_noalloc builds its tables in its own scratch."""
    import ctypes
    ny, nx, rows, cols, B = 600, 810, (-31, 63), (-43, 87), 3
    ks, full = _kernels(ny, nx, rows, cols, 3, 9)
    m = torch.as_tensor(np.random.default_rng(10).random((B, ny, nx)).astype(np.float32)).cuda()
    geo = nat.Geometry(ny=ny, nx=nx, k0r=rows[0], wr=rows[1], k0c=cols[0], wc=cols[1], nchan=1,
                       max_batch=B, max_kernels=3)
    chans = (ctypes.c_int * 1)(0)
    want = engine.socs_image(m, ks, pack_real=False)
    for _ in range(2):
        out = torch.empty_like(m)
        nat.check(nat.load().oi_socs_image_noalloc(ctypes.byref(geo), nat.ptr(m), nat.OI_FIELD_REAL, 1,
                                                   chans, B, nat.ptr(ks.win), 3, nat.ptr(out), nat.stream()))
        assert torch.equal(out, want)
