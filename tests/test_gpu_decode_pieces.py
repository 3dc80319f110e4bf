"""Decoded masks around the pieces of the decode kernels (4 pixels a lane, 1024
a pass, 8192 a workgroup): exact."""
import numpy as np
import pytest
import torch

from opticalimaging_amd import engine

pytestmark = pytest.mark.gpu

COUNTS = [3, 4, 5, 32, 36, 1020, 1024, 1028, 8188, 8191, 8192, 8193, 8224, 16384, 3 * 8192 + 1061]


@pytest.mark.parametrize("count", COUNTS)
def test_decode(gpu, count):
    rng = np.random.default_rng(count)
    codes = rng.integers(0, 6, count).astype(np.uint8)
    levels = (0.5, -1.0, 2.25, 7.0)
    out = engine.decode_mask_codes(torch.as_tensor(codes).cuda(), levels)
    assert np.array_equal(out.cpu().numpy(), np.array(levels + (0.0, 0.0), np.float32)[codes])
    bits = codes & 1
    out = engine.decode_mask_bits(torch.as_tensor(np.packbits(bits)).cuda(), (-3.0, 0.125), count)
    assert np.array_equal(out.cpu().numpy(), np.array((-3.0, 0.125), np.float32)[bits])
