"""The pupil crop from a windowed spectrum (the image's own window where it
holds the crop, else one of the crop's) against the crop of the full spectrum:
even and odd grids, one to three live channels out of several, windows that just
hold the crop and that miss it by one.  The unit circle is the same entry for
entry; values are two float32 transforms of the same field, whose rounding stays
below 4 log2(ny nx) 2^-24 of the largest."""
import math

import pytest
import torch

from opticalimaging_amd import _native as nat
from opticalimaging_amd import engine
from opticalimaging_amd.Scatter import full_spectrum, pupil_image

pytestmark = pytest.mark.gpu

CASES = [(64, 64, 3.6, 3.6, 1, (0,), True), (81, 135, 5.2, 9.7, 3, (0, 2), False),
         (160, 96, 11.0, 4.0, 3, (1, 2), False), (128, 125, 7.99, 6.01, 2, (1,), True),
         (100, 90, 2.5, 0.7, 3, (0, 1, 2), False)]


@pytest.mark.parametrize("ny,nx,px,py,cin,live,real", CASES)
@pytest.mark.parametrize("room", [-1, 0, 3, None])
def test_crop(gpu, ny, nx, px, py, cin, live, real, room):
    gen = torch.Generator(device="cuda").manual_seed(ny * nx)
    h = torch.zeros((ny, nx, cin), dtype=torch.complex64, device="cuda")
    for c in live:
        v = torch.randn((ny, nx), dtype=torch.complex64, device="cuda", generator=gen)
        h[..., c] = v.real if real else v
    enc = engine.field_encoding(h)
    tens, kind, c_in, chans = enc
    spectrum = None
    if room is not None:                       # a window of room entries past the crop
        oy, ox = int(py) + 3 + room, int(px) + 3 + room
        plan = engine.Plan(ny=ny, nx=nx, k0r=-oy, wr=2 * oy, k0c=-ox, wc=2 * ox + 1, nchan=len(chans),
                           max_kernels=1)
        spec = torch.empty((len(chans), 2 * oy, 2 * ox + 1), dtype=torch.complex64, device="cuda")
        cptr, keep = nat.int_array(chans)
        nat.check(nat.load().oi_spectrum_window(plan.handle, nat.ptr(tens), kind, c_in, cptr, 1,
                                                nat.ptr(spec), nat.stream()))
        spectrum = (spec, -oy, -ox)
    got = pupil_image(h, px, py, encoding=enc, spectrum=spectrum)
    ref = pupil_image(h, px, py, hk=full_spectrum(h, px, py))
    assert got.shape == ref.shape
    assert torch.equal(torch.isnan(got.real), torch.isnan(ref.real))
    assert bool(torch.isnan(got.real).any()) and not bool(torch.isnan(got.imag).any())
    err = (got - ref).abs().nan_to_num().max() / ref.abs().nan_to_num().max()
    assert err <= 4 * math.log2(ny * nx) * 2.0 ** -24, float(err)


def test_crop_refuses_a_short_window(gpu):
    t = torch.zeros(4096, dtype=torch.complex64, device="cuda")
    cptr, keep = nat.int_array([0])
    for k0r, wr, k0c, wc in ((-4, 10, -5, 10), (-5, 9, -5, 10), (-5, 10, -4, 10), (-5, 10, -5, 9)):
        with pytest.raises(ValueError):
            nat.check(nat.load().oi_pupil_crop(nat.ptr(t), 1, k0r, wr, k0c, wc, cptr, 1, 64, 64, 2.5, 2.5,
                                               5, 5, nat.ptr(t), nat.stream()))
