"""Compress and decompress where their chunk paths change, against the oracle
(byte-identical streams, bit-identical values): rates on both sides of a byte
slice (7 | 8, 15 | 16) and mixed within a chunk, extents whose chunks are runs
of whole blocks and extents that wrap, are cut or have rows shorter than a
chunk, and payloads that outgrow a wave's staging area early, late or in part."""
import numpy as np
import pytest

from tests.helpers import gpu_compress, gpu_decompress

pytestmark = pytest.mark.gpu

SHAPES = [(1, (0, 0, 0), 511), (1, (0, 0, 0), 512), (1, (0, 0, 0), 16384 + 2048 + 3), (1, (0, 0, 0), 70001)]
SHAPES += [(2, d, 0) for d in [(4, 3, 2), (60, 9, 5), (64, 8, 3), (64, 12, 2), (68, 17, 2), (128, 16, 9), (516, 20, 3), (576, 24, 2)]]
SHAPES += [(3, d, 0) for d in [(4, 5, 3), (28, 5, 7), (32, 4, 8), (32, 6, 4), (36, 9, 5), (64, 32, 12), (100, 36, 17)]]


def _values(n, dtype, seed, bits):
    """Steps of up to 2^bits[k] codes in runs of 48 values: with a bound of 0.5 the codes are the values."""
    r = np.random.default_rng(seed)
    top = np.repeat(r.choice(np.asarray(bits), -(-n // 48)), 48)[:n]
    step = np.floor(r.random(n) * 2.0 ** top) * r.choice([-1, 1], n)
    x = np.cumsum(step)
    return (x - np.round(x / 2.0**30) * 2.0**30).astype(dtype)   # codes stay below 2^31


def _check(oracle, x, eb, mode, dim, dims):
    want = oracle.compress(x, eb, mode, dim, dims)
    got = gpu_compress(x, eb, mode, dim, dims)
    assert got == want
    y = gpu_decompress(want, x.size, x.dtype, eb, mode, dim, dims)
    ref = oracle.decompress(want, x.size, x.dtype, eb, mode, dim, dims)
    iv = np.uint64 if x.dtype == np.float64 else np.uint32
    assert np.array_equal(y.view(iv), ref.view(iv))


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}D-{s[2] or 'x'.join(map(str, s[1]))}")
def test_rates_and_extents(device, oracle, shape, dtype):
    dim, dims, n = shape
    n = n or dims[0] * dims[1] * dims[2]
    for k, bits in enumerate(([0, 3, 6], [6, 7], [7, 8], [0, 7, 14], [14, 15], [3, 16, 24], [0, 30])):
        x = _values(n, dtype, 100 * k + n, bits)
        for mode in (0, 1, 2):
            _check(oracle, x, 0.5, mode, dim, dims)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_staging_area_overflows(device, oracle, dim, dtype):
    dims = {1: (0, 0, 0), 2: (192, 72, 3), 3: (96, 24, 18)}[dim]
    n = 41472
    for k, (low, high) in enumerate([(22, 22), (2, 26), (26, 2), (12, 12)]):
        bits = [low] * 20 + [high] * 20      # the first and the second half of a wave's chunks
        r = np.random.default_rng(k)
        top = np.repeat(np.resize(bits, -(-n // 128)), 128)[:n]
        x = (np.floor(r.random(n) * 2.0 ** top) * r.choice([-1, 1], n)).astype(dtype)
        for mode in (0, 1, 2):
            _check(oracle, x, 0.5, mode, dim, dims)


def _batch(P, torch, direction, rows):
    """rows: (in, out, values, capacity, bound, dim, dims, type, mode); the batch kernels' tiles are full ones."""
    with P.BatchPlan([P.batch_item(*r) for r in rows], direction) as plan:
        plan.execute()
        sizes, _ = plan.results()
    torch.cuda.synchronize()
    return sizes


# Values on both sides of each step of the tile shapes, of the longest header that a batch and a single call sum
# without a pass over it (16 and 256 KiB), and a few in between.
LINES = [(1, n + k) for n in (1, 2048, 65536, 524288, 1048576, 3145728, 6291456, 8388608) for k in (0, 1)]
LINES += [(3, (128, 64, z)) for z in (64, 65, 128, 129, 384, 385)] + [(3, (256, 128, 197)), (3, (256, 256, 256)), (3, (256, 256, 257))]
LINES += [(2, (1000, 1048, 1)), (2, (2048, 512, 1)), (2, (2044, 1537, 2)), (2, (4096, 4096, 1)), (2, (4096, 4097, 1))]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("line", LINES, ids=lambda s: f"{s[0]}D-{s[1]}")
def test_tile_shapes(device, oracle, line, dtype):
    import torch
    from cuszp_amd import pycuSZp as P

    dim, dims = line if line[0] > 1 else (1, (0, 0, 0))
    n = line[1] if dim == 1 else dims[0] * dims[1] * dims[2]
    r = np.random.default_rng(n)
    x = np.cumsum(r.integers(-5, 6, n)).astype(dtype)
    x[r.integers(0, n, n // 300 + 1)] += 5000
    t, typ = torch.from_numpy(x).cuda(), int(dtype == np.float64)
    for mode in (0, 1, 2):
        cap = P.max_compressed_size(n, dim, dims, typ, mode)
        one, two = torch.zeros(cap, dtype=torch.uint8, device="cuda"), torch.zeros(cap, dtype=torch.uint8, device="cuda")
        size = P.compress_ex(t, one, cap, n, 0.5, dim, dims, typ, mode)
        assert _batch(P, torch, P.BATCH_COMPRESS, [(t, two, n, cap, 0.5, dim, dims, typ, mode)]) == [size]
        assert torch.equal(one, two)
        if n <= 1 << 20:
            assert one[:size].cpu().numpy().tobytes() == oracle.compress(x, 0.5, mode, dim, dims)
        y, z = torch.full_like(t, float("nan")), torch.full_like(t, float("nan"))
        P.decompress_ex(y, one, n, size, 0.5, dim, dims, typ, mode)
        _batch(P, torch, P.BATCH_DECOMPRESS, [(one, z, n, size, 0.5, dim, dims, typ, mode)])
        assert torch.equal(y, t) and torch.equal(z, t)   # the codes are the values


@pytest.mark.parametrize("dim,dims,n", [(1, (0, 0, 0), 98304), (1, (0, 0, 0), 9 << 20), (3, (64, 64, 36), 147456), (2, (4096, 4104, 1), 4096 * 4104)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_any_header_byte(device, oracle, dim, dims, n, mode):
    """Streams that no compressor wrote: all 256 header bytes of outlier mode, all rates else, any payload."""
    r = np.random.default_rng(n + mode)
    nb = n // (32 if dim == 1 else 64)
    unit = 4 if dim == 1 else 8
    head = r.integers(0, 256 if mode == 2 else 32, nb, dtype=np.uint8)
    head[r.random(nb) < 0.9] = 0   # most of a long stream stays short
    if n < 1 << 20:
        head = r.permutation(np.resize(np.arange(256 if mode == 2 else 32, dtype=np.uint8), nb))
    R = (head & 31).astype(np.int64) if mode == 2 else head.astype(np.int64)
    sel = (head >> 7).astype(np.int64) if mode == 2 else 0
    size = np.where((R > 0) | (sel > 0), unit + unit * R, 0) + sel * (((head >> 5) & 3).astype(np.int64) + 1)
    pad = -(-n // 32768) * 1024 - nb if dim == 1 else -nb % 4
    cmp = head.tobytes() + bytes(pad) + r.integers(0, 256, int(size.sum()), dtype=np.uint8).tobytes()
    y = gpu_decompress(cmp, n, np.float32, 0.5, mode, dim, dims)
    ref = oracle.decompress(cmp, n, np.float32, 0.5, mode, dim, dims)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


# Offsets past 32 bits from a chunk's origin (general path, wide and narrow), the last extents inside them, narrow
# arrays of every width, rows whose last block is half outside with a single row below.
@pytest.mark.parametrize("dim,dims", [(2, (44739244, 3, 1)), (2, (16777212, 9, 1)), (2, (16777220, 9, 1)), (3, (4, 1048576, 5)), (3, (4, 1048572, 5)),
                                      (3, (8196, 4095, 5))] +
                         [(d, (x, 17, 5)) for d in (2, 3) for x in range(4, 76, 8)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_ragged_offsets(device, oracle, dim, dims, dtype):
    n = dims[0] * dims[1] * dims[2]
    r = np.random.default_rng(dims[0])
    x = (np.arange(n) * 7 % 1001 + r.integers(-9, 10, n)).astype(dtype)
    for mode in (0, 2) if n < 1 << 20 else (2,):
        want = oracle.compress(x, 0.5, mode, dim, dims, nthreads=oracle.max_threads())
        assert gpu_compress(x, 0.5, mode, dim, dims) == want
        assert np.array_equal(gpu_decompress(want, n, dtype, 0.5, mode, dim, dims), x)
