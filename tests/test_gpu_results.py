"""Lengths and statuses that the kernels leave in host memory: each call sees its
own, errors are seen once, and a plan's replays are independent of each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stream(P, torch, n, mode=1):
    t = torch.from_numpy(np.random.default_rng(n).normal(0, 100, n).astype(np.float32)).cuda()
    cap = P.max_compressed_size(n, 1, (0, 0, 0), 0, mode)
    out = torch.empty(cap, dtype=torch.uint8, device="cuda")
    return t, out, cap


@pytest.mark.parametrize("n", [1, 4097, 3 << 20])
def test_single_calls(device, oracle, n):
    import torch
    from cuszp_amd import pycuSZp as P

    t, out, cap = _stream(P, torch, n)
    want = len(oracle.compress(t.cpu().numpy(), 0.01, 1, 1, (0, 0, 0)))
    header = -(-n // 32768) * 1024
    y = torch.empty_like(t)
    for _ in range(2):
        assert P.compress_ex(t, out, cap, n, 0.01, mode=1) == want
        with pytest.raises(P.CuSZpError) as e:   # one byte short
            P.compress_ex(t, out, want - 1, n, 0.01, mode=1)
        assert e.value.status == 4
        assert P.compress_ex(t, out, want, n, 0.01, mode=1) == want   # and the next call is clean
        with pytest.raises(P.CuSZpError) as e:
            P.decompress_ex(y, out, n, max(header, want - 1), 0.01, mode=1)
        assert e.value.status == 5
        P.decompress_ex(y, out, n, want, 0.01, mode=1)
        assert (y - t).abs().max().item() <= 0.0102   # the bound, and 2 ulp of 500


@pytest.mark.parametrize("graph", [False, True])
def test_batch_replays(device, oracle, graph):
    import torch
    from cuszp_amd import pycuSZp as P

    ns = [1, 5000, 0, 70001, 300000]
    rows = [_stream(P, torch, n) if n else (None, None, 0) for n in ns]
    want = [len(oracle.compress(t.cpu().numpy(), 0.01, 1, 1, (0, 0, 0))) if n else 0 for n, (t, _, _) in zip(ns, rows)]
    caps = [c for _, _, c in rows]
    caps[3] = want[3] - 1   # this array does not fit
    items = [P.batch_item(t, o, n, c, 0.01, 1, (0, 0, 0), 0, 1) for n, (t, o, _), c in zip(ns, rows, caps)]
    with P.BatchPlan(items, P.BATCH_COMPRESS, graph=graph) as plan:
        for _ in range(3):
            plan.execute()
            sizes, st = plan.results(check=False)
            assert st == [0, 0, 0, 4, 0] and sizes == [want[0], want[1], 0, 0, want[4]]
            _, st = plan.results()   # seen once
            assert st == [0] * 5
    items[3] = P.batch_item(rows[3][0], rows[3][1], ns[3], want[3], 0.01, 1, (0, 0, 0), 0, 1)
    with P.BatchPlan(items, P.BATCH_COMPRESS, graph=graph) as plan:
        for _ in range(3):
            plan.execute()
            assert plan.results() == (want, [0] * 5)
