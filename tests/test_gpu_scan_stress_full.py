"""Forward progress of the inter-tile scan where tiles are full (8 waves of 8 chunks, f64
of 4) and where the offset pass runs with 1024 threads a workgroup (headers of
4 MiB and more), under the holds and claims of test_gpu_scan_stress.py, whose
arrays of 300,000 to 600,000 values have shorter tiles and whose headers are 320 KiB at most.

The arrays hold whole numbers and the bound is 0.5, so that the codes are the values."""
import numpy as np
import pytest

from tests.helpers import gpu_compress
from tests.test_gpu_scan_stress import AT_ONCE, HOLD, stress  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu

# more than 98,304 (f64 49,152) groups of 64 values: full tiles
TILES = [
    (1, (0, 0, 0), 16 << 20, np.float32, 1),
    (1, (0, 0, 0), (8 << 20) + 5, np.float64, 2),
    (2, (3000, 1999, 3), 0, np.float32, 2),
    (3, (256, 256, 128), 0, np.float64, 0),
]
# headers of more than 4 MiB
PASSES = [(1, (0, 0, 0), (128 << 20) + 1, np.float32, 1), (1, (0, 0, 0), (128 << 20) + 1, np.float32, 2), (3, (1024, 512, 516), 0, np.float32, 2)]


def _ids(c):
    return f"{c[0]}D-{np.dtype(c[3]).name}-m{c[4]}"


@pytest.mark.parametrize("knobs", [HOLD, AT_ONCE], ids=["hold", "steal-at-once"])
@pytest.mark.parametrize("case", TILES, ids=_ids)
def test_full_tile_claims(device, oracle, stress, case, knobs):  # noqa: F811
    from cuszp_amd import pycuSZp as P

    dim, dims, n, dtype, mode = case
    n = n or dims[0] * dims[1] * dims[2]
    r = np.random.default_rng(n)
    x = np.cumsum(r.integers(-5, 6, n)).astype(dtype)
    x[r.integers(0, n, n // 300)] += 5000
    want = oracle.compress(x, 0.5, mode, dim, dims, nthreads=oracle.max_threads())
    print(f"full tiles {_ids(case)} {knobs} n={n}", flush=True)
    stress(**knobs)
    got = gpu_compress(x, 0.5, mode, dim, dims)
    rc = P.scan_report()
    assert got == want
    assert rc["stolen"] and rc["claims"] > 0, rc


@pytest.mark.parametrize("knobs", [HOLD, AT_ONCE], ids=["hold", "steal-at-once"])
@pytest.mark.parametrize("case", PASSES, ids=_ids)
def test_long_header_claims(device, stress, case, knobs):  # noqa: F811
    import torch
    from cuszp_amd import pycuSZp as P

    dim, dims, n, dtype, mode = case
    n = n or dims[0] * dims[1] * dims[2]
    g = torch.Generator(device=device).manual_seed(n % 1000)
    t = torch.arange(n, device=device, dtype=torch.int32)
    t = (t * 7 % 1001 + torch.randint(-9, 10, (n,), generator=g, device=device, dtype=torch.int32)).to(torch.float32)
    cap = P.max_compressed_size(n, dim, dims, 0, mode)
    out = torch.empty(cap, dtype=torch.uint8, device=device)
    size = P.compress_ex(t, out, cap, n, 0.5, dim, dims, 0, mode)
    y = torch.full_like(t, float("nan"))
    print(f"long header {_ids(case)} {knobs} n={n}", flush=True)
    stress(**knobs)
    P.decompress_ex(y, out, n, size, 0.5, dim, dims, 0, mode)
    rd = P.scan_report()
    assert torch.equal(y, t)
    assert rd["stolen"] and rd["claims"] > 0, rd
