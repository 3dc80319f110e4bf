"""The two-pass coherent sum and its adjoint on the row-major column fields, at
every coarse size of the table (144, 256, 450, 512: groups of 12, 15 and 16
lanes), windows of few and many columns, odd and even, on and off the centre,
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
    (640, 512, (-60, 131), (-9, 17), 5, 1, 450),
    (512, 640, (-112, 225), (-107, 215), 3, 2, 450),
    (576, 576, (-128, 256), (-120, 231), 2, 1, 512),
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
