"""Lengths and errors that a lane's kernels leave in host memory: each request of a
batch sees its own, and the lane's next batch sees none of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 40_001, 700_000])   # headers that tiles sum up, and one that takes the offset pass
def test_a_lane_over_several_batches(device, oracle, n):
    import torch
    from cuszp_amd import pycuSZp as P

    x = torch.from_numpy(np.random.default_rng(n).normal(0, 100, n).astype(np.float32)).to(device)
    want = oracle.compress(x.cpu().numpy(), 1e-2, 1)
    c = torch.from_numpy(np.frombuffer(want, np.uint8).copy()).to(device)
    pool = torch.empty(64 << 20, dtype=torch.uint8, device=device)
    with P.Server(pool, lanes=1, max_batch=8) as S:
        for broken in (True, False, True, False, False):
            ids = [S.submit_compress(x, 1e-2, 1), S.submit_decompress(c, len(want), n, x.dtype, 1e-2, 1),
                   S.submit_decompress(c, len(want) - broken, n, x.dtype, 1e-2, 1), S.submit_compress(x, 1e-2, 1),
                   S.submit_decompress(c, len(want), n, x.dtype, 1e-2, 1)]
            got = {}
            while len(got) < len(ids):
                for rid, status, direction, off, nbytes in S.poll(wait=True):
                    got[rid] = (status, nbytes)
                    if status == 0:
                        out = pool[off:off + nbytes]
                        if direction == P.BATCH_COMPRESS:
                            assert out.cpu().numpy().tobytes() == want
                        else:
                            assert (out.view(torch.float32) - x).abs().max().item() <= 0.0101   # the bound, and 2 ulp of 500
                    S.release(rid)
            bad = (5, 0) if broken else (0, 4 * n)   # CUSZP_ERROR_CORRUPT_STREAM
            assert [got[i] for i in ids] == [(0, len(want)), (0, 4 * n), bad, (0, len(want)), (0, 4 * n)]
