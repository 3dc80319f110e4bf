"""Column fields of the two-pass sum where a plan holds those of a chunk of its
batch, or none: gradients that may read them only when all are there (coarse 100
and 128), images past coarse 512, and kernel sets of which one image's pass 4 GiB.
Images: the same squares in another order, K 2^-24 of the peak; gradients: twice
the transforms, as the other gradients of these lengths."""
import pytest
import torch

from opticalimaging_amd import engine
from test_gpu_dft_sizes import GRAD_TOL

pytestmark = pytest.mark.gpu


def _set(K, wr, wc, ny, nx, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    win = torch.randn((K, wr, wc), dtype=torch.complex64, device="cuda", generator=g)
    return engine.KernelSet(win, -(wr // 2), -(wc // 2), ny, nx), g


# the third needs 104 MB of column fields an image: six images in two chunks
@pytest.mark.parametrize("K,w,batch,coarse", [(5, 48, 3, 100), (7, 60, 2, 128), (1700, 60, 6, 128)])
def test_gradient_with_and_without_the_fields(gpu, K, w, batch, coarse):
    ks, gen = _set(K, w, w, 256, 256, K)
    plan = engine.plan_for(ks, 1, batch)
    assert (plan.info()["path"], plan.info()["lr"]) == (1, coarse)
    mask, target = torch.rand((2, batch, 256, 256), device="cuda", generator=gen)
    target = target * engine.socs_image(mask, ks, plan=plan, pack_real=False).mean()
    resid, grad, band = (torch.empty_like(mask) for _ in range(3))
    loss, blos = torch.zeros((2, 1), device="cuda")
    work = engine.adjoint_work(ks, batch, plan)
    assert engine.socs_residual_adjoint(mask, ks, target, resid, grad, work, loss=loss, plan=plan)
    ref = engine.socs_adjoint(mask, resid, ks, plan=plan, pack_real=False)   # forms its own fields
    assert (grad - ref).abs().max() <= GRAD_TOL * ref.abs().max()
    tband = engine.ilt_target_band(target, ks, work, plan=plan)
    engine.socs_band_residual_adjoint(mask, ks, tband, band, work, loss=blos, plan=plan)
    assert (band - ref).abs().max() <= 4 * GRAD_TOL * ref.abs().max()


def test_images_past_512_in_chunks(gpu):
    """85 MB an image, five or six of which a plan holds."""
    ks, gen = _set(64, 60, 288, 640, 640, 3)
    mask = torch.rand((8, 640, 640), device="cuda", generator=gen)
    info = engine.plan_for(ks, 1, 8).info()
    assert (info["path"], info["lr"]) == (2, 576)
    out = engine.socs_image(mask, ks, pack_real=False)
    ref = sum(engine.socs_image(mask[i:i + 1], ks, pack_real=False) * e for i, e in
              zip(range(8), torch.eye(8, device="cuda").reshape(8, 8, 1, 1)))
    assert (out - ref).abs().max() <= 64 * 2.0 ** -24 * ref.max()


def test_general_kernels_past_the_bound(gpu):
    """3500 kernels would need 4.6 GB an image past coarse 512."""
    ks, gen = _set(4, 60, 288, 640, 640, 4)
    mask = torch.rand((1, 640, 640), device="cuda", generator=gen)
    plan = engine.Plan(640, 640, ks.k0r, ks.wr, ks.k0c, ks.wc, max_kernels=3500)
    assert plan.info()["path"] == 0 and not plan.info()["direct"]
    out = engine.socs_image(mask, ks, plan=plan, pack_real=False)
    ref = engine.socs_image(mask, ks, pack_real=False)
    assert (out - ref).abs().max() <= 6e-6 * ref.max()      # other transforms
