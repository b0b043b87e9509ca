"""The grid reductions (value range, error figures, SSIM) where their shares of
the work change: array starts off a 16-byte boundary, a step of the figures'
loop more or less, several steps per workgroup, window tiles that are cut or
narrow, volumes of one window, and values far from zero.

Tolerance of the sums: the oracle adds n terms one after another in double, so
its own error is at most n * 2^-53 relative (5e-10 at the largest n here) plus
the device's, which adds in a tree: 1e-9."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SUMS = ("mse", "psnr", "norm_err", "norm_err_norm", "nrmse", "correlation")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [15, 4095, 4096, 4097, 1024 * 4096 + 4096 + 7])
def test_figures_edges(device, oracle, dtype, n):
    import torch
    from cuszp_amd import pycuSZp as P

    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n + 3) * 7 + 300).astype(dtype)
    y = (x + rng.uniform(-0.5, 0.5, n + 3)).astype(dtype)
    tx, ty = torch.from_numpy(x).to(device), torch.from_numpy(y).to(device)
    for ox, oy in ((0, 0), (1, 3)):
        got = P.quality(tx[ox:ox + n], ty[oy:oy + n])
        want = oracle.quality(x[ox:ox + n].copy(), y[oy:oy + n].copy())
        for k in ("range", "max_abs_err", "max_rel_err"):
            assert got[k] == want[k], k
        for k in SUMS:
            assert got[k] == pytest.approx(want[k], rel=1e-9), k


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dims", [(7, 7, 7), (8, 9, 10), (21, 90, 11), (69, 22, 7), (71, 23, 24), (140, 7, 12)])
@pytest.mark.parametrize("offset", [0.0, 5000.0])
def test_ssim_tiles(device, oracle, dtype, dims, offset):
    import torch
    from cuszp_amd import pycuSZp as P

    rng = np.random.default_rng(sum(dims))
    n = dims[0] * dims[1] * dims[2]
    x = (np.cumsum(rng.standard_normal(n)) * 0.1 + offset).astype(dtype)
    y = (x + rng.uniform(-0.05, 0.05, n)).astype(dtype)
    x[: n // 3] = x[0]      # windows of one value: range and variance 0
    got = P.ssim(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device), dims)
    assert got == pytest.approx(oracle.ssim(x, y, dims), rel=1e-9)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [2, 2047, 8192, 8193, 9_000_001])
def test_range_edges(device, oracle, dtype, n):
    import torch
    from cuszp_amd import pycuSZp as P

    x = np.random.default_rng(n).standard_normal(n + 3).astype(dtype)
    t = torch.from_numpy(x).to(device)
    for off in range(4):
        for at in (0, n // 2, n - 1):   # the extreme value anywhere in the share of any lane
            h = x[off:off + n].copy()
            h[at] = -1e6
            t[off + at] = -1e6
            assert P.value_range(t[off:off + n]) == (float(h.min()), float(h.max()))
            t[off + at] = float(x[off + at])


@pytest.mark.parametrize("scale", [1e-30, 1e-20, 1e20, 1e37])
def test_ssim_scales(device, oracle, scale):
    """Floats near both ends of their range: the window formula's products stay within double's."""
    import torch
    from cuszp_amd import pycuSZp as P

    dims = (40, 19, 13)
    r = np.random.default_rng(3)
    n = dims[0] * dims[1] * dims[2]
    x = (r.normal(1, 0.5, n) * scale).astype(np.float32)
    y = (x * (1 + 0.05 * r.normal(0, 1, n))).astype(np.float32)
    got = P.ssim(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device), dims)
    assert got == pytest.approx(oracle.ssim(x, y, dims), rel=1e-9)
