"""The per-image constant of the band loss from targets that start on a 16-byte
boundary (four pixels a load) and one float past it (one a load): the float64
sums differ in their order only, so the float32 losses differ by a rounding, and
both are the loss of the float64 image up to its own error (1e-5)."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import ILT
from test_gpu_dft_sizes import _image, _kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nx,half,batch", [(128, 128, 8, 3), (256, 512, 27, 1), (512, 256, 40, 2)])
def test_target_alignment(gpu, ny, nx, half, batch):
    ks, full = _kernels(ny, nx, (-half, 2 * half + 1), (-half, 2 * half + 1), 2, ny)
    ks.win /= 100.0
    rng = np.random.default_rng(nx)
    th = rng.standard_normal((batch, ny, nx)).astype(np.float32)
    T = rng.random((batch, ny, nx)).astype(np.float32)
    flat = torch.empty(T.size + 1, device="cuda")
    off = flat[1:].view(T.shape)
    off.copy_(torch.as_tensor(T))
    losses = []
    for target in (torch.as_tensor(T).cuda(), off):
        _, loss = ILT.ilt(torch.as_tensor(th).cuda(), target, ks, steps=1, lr=0.1)
        losses.append(float(loss[0]))
    m = 1 / (1 + np.exp(-th.astype(np.float64)))
    ref = sum(((_image(full / 100.0, m[b]) - T[b]) ** 2).sum() for b in range(batch))
    assert abs(losses[0] - losses[1]) <= 2.0 ** -22 * ref
    assert abs(losses[0] - ref) <= 1e-5 * ref
