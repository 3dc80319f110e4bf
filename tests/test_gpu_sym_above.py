"""oi_sym_above (is the smallest eigenvalue above a share of the trace) at the
edges of its 32-wide panels, against eigenvalues set a tenth of a percent above
and below the line (its rounding, about n eps of the trace, is 1e-6 of that),
and the decision it takes for engine.real_mask_kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _with_smallest(n, share, seed):
    rng = np.random.default_rng(seed)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    lam = 10.0 ** rng.uniform(-4, 0, n)
    rest = lam[1:].sum() if n > 1 else 0.0
    lam[0] = share / (1 - share) * rest if n > 1 else 1.0
    G = (Q * lam) @ Q.T
    return torch.as_tensor((G + G.T) / 2).cuda()


@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 63, 64, 65, 97, 240])
def test_line_is_where_it_says(gpu, n):
    from opticalimaging_amd.engine import _sym_above
    rel = 1e-7
    assert _sym_above(_with_smallest(n, rel * 1.001, n), rel)
    assert not _sym_above(_with_smallest(n, rel * 0.999, n), rel)


def test_not_positive_or_not_finite_is_not_above(gpu):
    from opticalimaging_amd.engine import _sym_above
    G = torch.eye(70, dtype=torch.float64, device="cuda")
    assert _sym_above(G, 1e-3)
    for bad in (-1.0, 0.0, float("nan")):
        for at in (0, 33, 69):
            H = G.clone()
            H[at, at] = bad
            assert not _sym_above(H, 1e-10)
    assert not _sym_above(torch.zeros_like(G), 1e-10)


@pytest.mark.parametrize("defocus", [0.0, 80.0])
@pytest.mark.parametrize("order", [12, 120])
def test_pairing_decision_is_the_eigenvalues(gpu, defocus, order):
    """The set that real_mask_kernels returns with and without the check."""
    from opticalimaging_amd import engine, workloads
    from opticalimaging_amd.DecomposeTCC_SOCS import socs_kernel_set
    src, proj, num = workloads.socs_1024_optics(order=order, grid_halfwidth=None)
    ks = socs_kernel_set(src, [1000.0, 1000.0], proj, defocus, num, [128, 128])
    with_check = engine.real_mask_kernels(ks)
    check, engine._sym_above = engine._sym_above, lambda *a: False
    try:
        without = engine.real_mask_kernels(ks)
    finally:
        engine._sym_above = check
    assert with_check.K == without.K
    assert (with_check is ks) == (without is ks)
