"""Shapes that AbbeSourceProblem.source_gradient takes besides one cotangent per
focus: no focus at all, and cotangents of more foci than the problem has."""
import pytest
import torch

from gpu_cases import annular, numerics, projector, scatter
from opticalimaging_amd import SMO, workloads

pytestmark = pytest.mark.gpu


def _problem(foci):
    proj = projector(M=1)
    proj.FocusRange = torch.tensor(foci, dtype=torch.float32)
    gen = torch.Generator().manual_seed(3)
    field = workloads.field_from_mask((torch.rand((64, 64), generator=gen) < 0.4).float().numpy())
    return SMO.abbe_source_problem(field.cuda(), annular(P=11), scatter(field.cuda(), 1000.0, 1000.0), proj,
                                   numerics(mode="scalar"))


def test_no_focus_gives_zeros(gpu):
    prob = _problem([])
    V = prob.V0.clone().requires_grad_(True)
    image = SMO.abbe_image_weighted(V, prob)
    assert image.shape == (0, 64, 64)
    # memory that the allocator hands out again
    used = [torch.full((prob.nsrc,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(256)]
    del used
    image.sum().backward()
    assert torch.equal(V.grad, torch.zeros_like(V))


def test_cotangents_of_more_foci(gpu):
    prob = _problem([0.0, 40.0])
    g = torch.randn((3, 64, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    assert torch.equal(prob.source_gradient(prob.V0, g), prob.source_gradient(prob.V0, g[:2]))
    for bad in (g[:1], g[:2, :63], g[:2].reshape(2, -1)):
        with pytest.raises(ValueError):
            prob.source_gradient(prob.V0, bad)
