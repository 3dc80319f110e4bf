"""CalculateAbbeImage through focus where the coarse grid is summed in two passes
(100 and 128): the kernel groups are the ones that the two-pass sum chooses (at
most 64 partial sums an image), and the foci in one launch chain are the foci one
by one (same squares in another order: K 2^-24 of the peak)."""
import pytest
import torch

from gpu_cases import numerics, projector, quasar, scatter
from opticalimaging_amd import CalculateAbbeImage, engine, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nx,foci,coarse", [(400, 400, 4, 100), (480, 300, 5, 128), (320, 320, 5, 75)])
def test_foci(gpu, ny, nx, foci, coarse):
    gen = torch.Generator().manual_seed(ny)
    field = workloads.field_from_mask((torch.rand((ny, nx), generator=gen) < 0.4).float().numpy()).cuda()
    src, sc, num = quasar(), scatter(field, 8.0 * nx, 8.0 * ny), numerics(mode="vector")

    def image(z):
        return CalculateAbbeImage(src, sc, projector(NA=1.35, n=1.44, M=1, foci=z), num)[0].Intensity
    zs = [30.0 * i - 40.0 for i in range(foci)]
    engine.PLANS.plans.clear()
    many = image(zs).reshape(foci, ny, nx)
    plan, = [p.info() for p in engine.PLANS.plans.values() if p.info()["max_batch"] == foci]
    assert plan["lr"] == coarse and plan["max_kernels"] * foci >= 2048
    # coarse 75 is summed in one pass, where 512 workgroups have four kernels each
    assert plan["max_groups"] <= 64 if coarse > 75 else plan["max_groups"] == -(-512 // foci)
    one = torch.cat([image([z]).reshape(1, ny, nx) for z in zs])
    assert (many - one).abs().max() <= plan["max_kernels"] * 2.0 ** -24 * one.max()
