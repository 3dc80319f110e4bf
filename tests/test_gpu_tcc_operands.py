"""The contraction's operand planes at the edges of their 64 x 32 tiles, in the
three precisions, against a float64 product.  Entries are sums of r products of
numbers near 1: split-bf16 drops the lo lo' term (2^-16 of a product, signs at
random) and rounds to float32, float32 sums r terms, float64 rounds once."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

PRECISIONS = {0: 2.0 ** -16, 1: 2.0 ** -24, 2: 0.0}


@pytest.mark.parametrize("code", PRECISIONS)
@pytest.mark.parametrize("M,nsrc,ncomp", [(1, 1, 1), (49, 15, 1), (64, 16, 2), (65, 33, 1), (190, 31, 3), (257, 64, 1)])
def test_planes(gpu, M, nsrc, ncomp, code):
    from opticalimaging_amd.CalculateTCCMatrix import tcc_contract
    gen = torch.Generator().manual_seed(M)
    G = torch.randn((ncomp, nsrc, M), dtype=torch.complex64, generator=gen)
    w = torch.rand(nsrc, generator=gen) + 0.1
    out = tcc_contract(G.cuda(), w.cuda(), 0.5, code).cpu().to(torch.complex128)
    A = (G.to(torch.complex128) * w.double().sqrt()[None, :, None]).reshape(-1, M)
    ref = 0.5 * A.T @ A.conj()
    r = nsrc * ncomp
    tol = 4 * math.sqrt(r) * PRECISIONS[code] + 2.0 ** -22      # sqrt(w) and G rounded once each
    if code == 1:
        tol += r * 2.0 ** -24
    assert (out.reshape(M, M) - ref).abs().max() <= tol * ref.abs().max()
