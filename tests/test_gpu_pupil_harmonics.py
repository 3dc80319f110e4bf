"""The wavefront sum with only some of the harmonics 0..5 of theta present (an
absent one is passed over), on oi_zernike.  The device sums in float64 and
rounds once: 2^-24 of the value, taken twice over."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

# one cosine and one sine term (0-based) of each harmonic, and sets that leave gaps
TERMS = [[], [0], [8, 36], [1], [14], [4], [21], [9], [10], [16], [17], [25], [26], [3, 26],
         [2, 10, 25], list(range(37))]


@pytest.mark.parametrize("terms", TERMS, ids=str)
def test_present_harmonics_only(gpu, terms):
    from opticalimaging_amd import Projection
    rng = np.random.default_rng(len(terms))
    p = Projection()
    c = np.zeros(37, np.float32)
    c[terms] = rng.uniform(0.05, 1.0, len(terms))
    p.Aberration_Zernike = torch.tensor(c)
    rho = np.append(np.sqrt(rng.random(700)), [0.0, 1.0]).astype(np.float32)
    th = np.append(rng.uniform(-np.pi, np.pi, 700), [0.0, 0.5]).astype(np.float32)
    w = p.CalculateAberrationFast(torch.tensor(rho).cuda(), torch.tensor(th).cuda(), 0.0)
    ref = O.zernike_fringe(rho.astype(np.float64), th.astype(np.float64), c.astype(np.float64))
    assert np.max(np.abs(w.cpu().numpy() - ref)) <= 2.0 ** -23 * c.sum()
