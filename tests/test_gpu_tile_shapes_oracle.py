"""Compressed bytes of every tile shape against the oracle, for the array lengths at which
the shape changes. (test_tile_shapes compares the longer ones with a batch only, whose
tiles have the same shape; the batch here holds a long array too, so its tiles are full.)"""
import numpy as np
import pytest

from tests.test_gpu_chunk_paths import LINES

pytestmark = pytest.mark.gpu


def _size(line):
    return line[1] if line[0] == 1 else line[1][0] * line[1][1] * line[1][2]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("line", [v for v in LINES if _size(v) > 1 << 20], ids=lambda s: f"{s[0]}D-{s[1]}")
def test_long_lines(device, oracle, line, dtype):
    import torch
    from cuszp_amd import pycuSZp as P

    dim, dims = line if line[0] > 1 else (1, (0, 0, 0))
    n = _size(line)
    r = np.random.default_rng(n)
    x = np.cumsum(r.integers(-5, 6, n)).astype(dtype)
    x[r.integers(0, n, n // 300 + 1)] += 5000
    t, typ = torch.from_numpy(x).cuda(), int(dtype == np.float64)
    for mode in (0, 1, 2):
        cap = P.max_compressed_size(n, dim, dims, typ, mode)
        out = torch.zeros(cap, dtype=torch.uint8, device="cuda")
        size = P.compress_ex(t, out, cap, n, 0.5, dim, dims, typ, mode)
        assert out[:size].cpu().numpy().tobytes() == oracle.compress(x, 0.5, mode, dim, dims, nthreads=oracle.max_threads())


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_short_arrays_in_full_tiles(device, oracle, mode, dtype):
    import torch
    from cuszp_amd import pycuSZp as P

    typ = int(dtype == np.float64)
    shapes = [(1, (0, 0, 0), 16 << 20), (1, (0, 0, 0), 1), (1, (0, 0, 0), 65537), (2, (1000, 1048, 1), 1048000), (3, (128, 64, 65), 128 * 64 * 65),
              (1, (0, 0, 0), 524289)]
    xs, ts, outs, items = [], [], [], []
    for dim, dims, n in shapes:
        r = np.random.default_rng(n)
        x = np.cumsum(r.integers(-5, 6, n)).astype(dtype)
        x[r.integers(0, n, n // 300 + 1)] += 5000
        cap = P.max_compressed_size(n, dim, dims, typ, mode)
        xs.append(x)
        ts.append(torch.from_numpy(x).cuda())
        outs.append(torch.zeros(cap, dtype=torch.uint8, device="cuda"))
        items.append(P.batch_item(ts[-1], outs[-1], n, cap, 0.5, dim, dims, typ, mode))
    with P.BatchPlan(items, P.BATCH_COMPRESS) as plan:
        plan.execute()
        sizes, _ = plan.results()
    for (dim, dims, n), x, o, size in zip(shapes, xs, outs, sizes):
        assert o[:size].cpu().numpy().tobytes() == oracle.compress(x, 0.5, mode, dim, dims, nthreads=oracle.max_threads())
