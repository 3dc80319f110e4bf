"""oi_coherent_sets (one spectrum, several kernel sets) against oi_coherent_image
on each set: one-pass plans that take the sets in chains of max_batch (with a
remainder), two-pass, generic and direct plans that take them one by one.  Same
terms in another summation order: float32 sums of up to 3 K squares, compared at
3 K 2^-24 of the largest pixel."""
import pytest
import torch

from opticalimaging_amd import _native as nat
from opticalimaging_amd import engine

pytestmark = pytest.mark.gpu

# (ny, nx), window, band, channels, max_batch, sets
CASES = [((128, 128), (21, 23), (11, 12), 1, 5, 5),      # one-pass, one chain
         ((128, 160), (31, 29), (17, 15), 3, 3, 7),      # one-pass, 3 + 3 + 1, products
         ((256, 256), (80, 84), (50, 48), 2, 2, 3),      # one-pass kernel of L = 100
         ((512, 512), (101, 99), (70, 66), 1, 2, 3),     # two-pass: one by one
         ((64, 64), (40, 40), (40, 40), 2, 4, 2)]        # direct: one by one


@pytest.mark.parametrize("grid,win,band,nchan,batch,sets", CASES)
def test_sets_match_single(gpu, grid, win, band, nchan, batch, sets):
    (ny, nx), (wr, wc) = grid, win
    K, lib = 11, nat.load()
    g = torch.Generator(device="cuda").manual_seed(ny + wr)
    spec = torch.randn((nchan, wr, wc), dtype=torch.complex64, device="cuda", generator=g)
    kern = torch.randn((sets, K, wr, wc), dtype=torch.complex64, device="cuda", generator=g)
    # every kernel inside one band, as shifted pupils are
    kern[..., band[0]:, :] = 0
    kern[..., :, band[1]:] = 0
    kw = dict(ny=ny, nx=nx, k0r=-(wr // 2), wr=wr, k0c=-(wc // 2), wc=wc, nchan=nchan, band_r=band[0],
              band_c=band[1], max_kernels=K)
    many, one = engine.Plan(max_batch=batch, **kw), engine.Plan(max_batch=1, **kw)
    out = torch.full((sets, ny, nx), float("nan"), device="cuda")
    nat.check(lib.oi_coherent_sets(many.handle, nat.ptr(spec), sets, nat.ptr(kern), K, nat.ptr(out),
                                   nat.stream()))
    ref = torch.empty_like(out)
    for s in range(sets):
        nat.check(lib.oi_coherent_image(one.handle, nat.ptr(spec), 1, nat.ptr(kern[s]), K,
                                        nat.ptr(ref[s]), nat.stream()))
    err = (out - ref).abs().max() / ref.max()
    assert err <= 3 * K * 2.0 ** -24, float(err)


def test_sets_refuse_bad_counts(gpu):
    plan = engine.Plan(ny=128, nx=128, k0r=-4, wr=9, k0c=-4, wc=9, band_r=9, band_c=9, max_kernels=2)
    t = torch.zeros(1 << 16, device="cuda")
    for sets, K in ((0, 1), (1, 0), (1, 3)):
        with pytest.raises(ValueError):
            nat.check(nat.load().oi_coherent_sets(plan.handle, nat.ptr(t), sets, nat.ptr(t), K,
                                                  nat.ptr(t), nat.stream()))
