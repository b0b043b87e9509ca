"""The error figures and SSIM at their limits: f64 values near the ends of double's
range, where products of sums or of means leave it although the results do not,
and volumes with few windows along two axes."""
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


@pytest.mark.parametrize("scale", [1e-150, 1e150, 3e151, 3e152, 6e152])
@pytest.mark.parametrize("offset", [0.0, 1.0])
@pytest.mark.parametrize("dims", [(7, 7, 7), (40, 19, 13), (9, 70, 11)])
def test_ssim_far_deviations(device, oracle, scale, offset, dims):
    """Deviations whose own squares sum to less than double's largest value, while
    those of sums of many of them do not; the same tolerance as near 1."""
    import torch
    from cuszp_amd import pycuSZp as P

    r = np.random.default_rng(11)
    n = dims[0] * dims[1] * dims[2]
    x = (r.uniform(-1.7, 1.7, n) + offset) * scale
    y = x * (1 + 0.05 * r.uniform(-1.7, 1.7, n))
    want = oracle.ssim(x, y, dims)
    assert np.isfinite(want)
    assert P.ssim(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device), dims) == pytest.approx(want, rel=1e-9)
    x[n // 2] = np.inf   # no window's values by themselves
    assert np.isnan(P.ssim(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device), dims)) == np.isnan(oracle.ssim(x, y, dims))


# On both sides of the lines between tiles and a thread per window (9 slices in a row; 65,536 windows), the few
# windows along any two of the axes, and more windows than the largest grid has threads.
THIN = [(7, 7, 1505), (7, 7, 4005), (7, 9, 3005), (9, 9, 6005), (13, 13, 3755), (8, 21, 7505), (22, 7, 7507), (7, 60005, 7), (60006, 8, 7),
        (30005, 7, 9), (7, 7, 140005), (21, 7, 17505), (9, 7, 400005)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims", THIN)
def test_ssim_thin_volumes(device, oracle, dtype, dims):
    """Tolerance: both sides add up to 400,000 windows' values near 1 in double, 5e-11 at most."""
    import torch
    from cuszp_amd import pycuSZp as P

    r = np.random.default_rng(sum(dims))
    n = dims[0] * dims[1] * dims[2]
    x = (np.cumsum(r.standard_normal(n)) * 0.1).astype(dtype)
    y = (x + r.uniform(-0.05, 0.05, n)).astype(dtype)
    x[: n // 3] = x[0]      # windows of one value
    got = P.ssim(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device), dims)
    assert got == pytest.approx(oracle.ssim(x, y, dims), rel=1e-9)
