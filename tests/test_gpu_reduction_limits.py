"""The error figures and SSIM of f64 values near the ends of double's range, where
products of sums or of means leave it although the results do not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mean", [1e-140, 1e150, 2e154, -1e155])
@pytest.mark.parametrize("n", [15, 2048, 2049, 70001])
def test_figures_far_means(device, oracle, mean, n):
    """Means whose squares overflow, deviations (1e-6 of the mean) whose squares do not.

    Both sides find a mean to n * 2^-53 of its size, 8e-6 of the deviations at
    the largest n; the correlation sees the square of that, 6e-11: 1e-9."""
    import torch
    from cuszp_amd import pycuSZp as P

    r = np.random.default_rng(n)
    u = r.standard_normal(n)
    x = mean * (1 + 1e-6 * u)
    y = mean * (1 + 1e-6 * (u + 0.1 * r.standard_normal(n)))
    got = P.quality(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device))
    want = oracle.quality(x, y)
    for k in ("range", "max_abs_err", "max_rel_err"):
        assert got[k] == want[k], k
    for k in ("mse", "nrmse", "correlation"):
        assert np.isfinite(want[k]) and got[k] == pytest.approx(want[k], rel=1e-9), k
