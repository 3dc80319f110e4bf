"""oi_coherent_sets on plans of the generic kernels (a coarse grid of the caller's
choice; a grid that is its own coarse grid): the sets are summed one by one in the
kernel groups of a one-image plan, bit for bit, however many sets the plan is for."""
import pytest
import torch

from opticalimaging_amd import _native as nat
from opticalimaging_amd import engine

pytestmark = pytest.mark.gpu


# grid, window, band, coarse grid (0, 0: the library's), kernels, max_batch, sets
@pytest.mark.parametrize("grid,win,band,coarse,K,batch,sets", [
    ((256, 128), (43, 41), (23, 22), (48, 60), 150, 5, 7), ((240, 200), (109, 85), (58, 45), (120, 96), 70, 16, 3),
    ((64, 60), (40, 40), (40, 40), (0, 0), 90, 9, 2), ((128, 512), (21, 23), (11, 12), (24, 32), 3, 2, 2)])
def test_groups_of_one_image(gpu, grid, win, band, coarse, K, batch, sets):
    (ny, nx), (wr, wc), lib = grid, win, nat.load()
    g = torch.Generator(device="cuda").manual_seed(ny + wr)
    spec = torch.randn((2, wr, wc), dtype=torch.complex64, device="cuda", generator=g)
    kern = torch.randn((sets, K, wr, wc), dtype=torch.complex64, device="cuda", generator=g)
    kern[..., band[0]:, :] = 0
    kern[..., :, band[1]:] = 0
    kw = dict(ny=ny, nx=nx, k0r=-(wr // 2), wr=wr, k0c=-(wc // 2), wc=wc, nchan=2, band_r=band[0],
              band_c=band[1], lr=coarse[0], lc=coarse[1], max_kernels=K)
    many, one = engine.Plan(max_batch=batch, **kw), engine.Plan(max_batch=1, **kw)
    assert many.info()["path"] == 0
    assert many.info()["direct"] or (many.info()["lr"], many.info()["lc"]) == coarse
    out, ref = (torch.full((sets, ny, nx), float("nan"), device="cuda") for _ in range(2))
    nat.check(lib.oi_coherent_sets(many.handle, nat.ptr(spec), sets, nat.ptr(kern), K, nat.ptr(out), nat.stream()))
    for s in range(sets):
        nat.check(lib.oi_coherent_image(one.handle, nat.ptr(spec), 1, nat.ptr(kern[s]), K, nat.ptr(ref[s]),
                                        nat.stream()))
    assert torch.isfinite(ref).all() and torch.equal(out, ref)
