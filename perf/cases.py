"""The work that programs built on this library have it do, as cases that can be timed.

A case is one pass through the public Python entry points (cuszp_amd/pycuSZp.py, which call the C ABI
directly): single arrays in both directions, small to 4 GiB, 1D / 2D / 3D, fixed / plain / outlier,
float32 / float64, extents that fit the blocks and extents that do not; a relative bound with the value
range taken on the device; a batch of arrays of mixed sizes through a captured plan; and the quality report
of a reconstruction.

The data are those of the benchmark and the tests: "field" (a sum of eight sinusoids with noise, some runs
zeroed), "grf" (a Gaussian random field of spectrum k^-11/3 with 0.1 % spikes) and "weight" (normal
values). Everything is made on the GPU from the seed.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from cuszp_amd import pycuSZp as P

DEV = "cuda:0"
FIELD_FREQ = (1e-6, 1e-3)      # cycles per element
WEIGHT_SIGMA = 0.02
# Stream bytes per value that these data give, by mode and bound (measured once on 16 Mi values): the share
# of work() that depends on the data.
STREAM_BYTES = {
    ("field", "plain", 1e-2): 0.42, ("field", "plain", 1e-3): 0.74, ("field", "plain", 1e-4): 1.07,
    ("field", "outlier", 1e-2): 0.21, ("field", "outlier", 1e-3): 0.26, ("field", "outlier", 1e-4): 0.43,
    ("grf", "plain", 1e-2): 0.12, ("grf", "plain", 1e-3): 0.45, ("grf", "plain", 1e-4): 0.83,
    ("grf", "outlier", 1e-2): 0.12, ("grf", "outlier", 1e-3): 0.41, ("grf", "outlier", 1e-4): 0.76,
    ("weight", "fixed", 1e-3): 0.79,
}


def _single(name, op, dim, mode, dtype, data, bound, x, y=0, z=0):
    return {"name": name, "op": op, "dim": dim, "mode": mode, "dtype": dtype, "data": data, "bound": bound,
            "x": x, "y": y, "z": z}


def listed():
    return [
        # a short array through the blocking calls, as a program that compresses message by message makes
        # them: 16,001 values (64 KiB, the smallest request of the serving trace); calls and launches count
        _single("small_1d_plain_f32", "roundtrip", 1, "plain", "f32", "field", 1e-3, 16_001),
        # one variable of a simulation's dump with a bound relative to its range: value range on the
        # device, then compression (64 MiB, with zeroed runs)
        _single("rel_1d_plain_f32", "compress_rel", 1, "plain", "f32", "field", 1e-3, 16_777_216),
        # reading back a ragged array of doubles (48 MB of values)
        _single("read_1d_outlier_f64", "decompress", 1, "outlier", "f64", "field", 1e-4, 6_000_011),
        # the volume workload, each direction by itself: 512^3 values, outlier mode
        _single("write_3d_outlier_f32", "compress", 3, "outlier", "f32", "grf", 1e-4, 512, 512, 512),
        _single("read_3d_outlier_f32", "decompress", 3, "outlier", "f32", "grf", 1e-4, 512, 512, 512),
        # a volume whose extents fit neither the blocks nor a run of blocks, written and read back
        _single("ragged_3d_plain_f32", "roundtrip", 3, "plain", "f32", "grf", 1e-3, 600, 450, 150),
        # a stack of slices, likewise: 375 blocks to a row, a last row of blocks that is cut
        _single("ragged_2d_outlier_f32", "roundtrip", 2, "outlier", "f32", "grf", 1e-3, 3000, 1999, 16),
        # a matrix of weights in doubles, no prediction
        _single("matrix_2d_fixed_f64", "roundtrip", 2, "fixed", "f64", "weight", 1e-3, 8192, 8192, 1),
        # a checkpoint's tensors or a dump's variables in one call per direction: 256 arrays of 1,024 to
        # 16 Mi values, half weights and half fields, 30 % doubles, as one captured plan
        {"name": "batch_write_256", "op": "batch_compress", "count": 256, "largest": 1 << 24, "spec": 3},
        {"name": "batch_read_256", "op": "batch_decompress", "count": 256, "largest": 1 << 24, "spec": 3},
        # the large array of the headline benchmark: 4 GiB written and read back
        _single("large_1d_plain_f32", "roundtrip", 1, "plain", "f32", "field", 1e-3, 1 << 30),
        # the report that follows a trial of bounds: error figures and windowed SSIM of a volume
        _single("report_3d_f32", "report", 3, "outlier", "f32", "grf", 1e-3, 300, 280, 260),
    ]


def draw(rng: random.Random):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["roundtrip", "roundtrip", "compress", "decompress", "compress", "decompress", "compress_rel",
                     "batch_compress", "batch_decompress", "report"])
    if op.startswith("batch"):
        return {"op": op, "count": log_int(16, 256), "largest": log_int(1 << 17, 1 << 24), "spec": rng.randrange(1 << 20)}
    dtype = "f32" if rng.random() < 0.7 else "f64"
    if op == "report":
        n = log_int(1 << 16, 1 << 25)
        z, y = rng.randint(16, 200), log_int(16, 400)
        return _draw_single(op, 3, "outlier", dtype, "grf", 1e-3, max(8, n // (y * z) // 4 * 4), y, z)
    dim = rng.choice([1, 1, 2, 3])
    if dim == 1:
        data = rng.choice(["field", "field", "weight"])
        mode = "fixed" if data == "weight" else rng.choice(["plain", "outlier"])
        bound = 1e-3 if data == "weight" else rng.choice([1e-2, 1e-3, 1e-4])
        return _draw_single(op, 1, mode, dtype, data, bound, log_int(1024, (1 << 29) // (2 if dtype == "f64" else 1)))
    n = log_int(1 << 14, (1 << 27) // (2 if dtype == "f64" else 1))
    data = rng.choice(["grf", "grf", "weight"])
    mode = "fixed" if data == "weight" else rng.choice(["plain", "outlier"])
    bound = 1e-3 if data == "weight" else rng.choice([1e-2, 1e-3, 1e-4])
    side = n ** (1.0 / dim)
    y = max(1, int(side * math.exp(rng.uniform(-0.7, 0.7))))
    z = max(1, int(side * math.exp(rng.uniform(-0.7, 0.7)))) if dim == 3 else rng.choice([1, 1, rng.randint(2, 32)])
    x = max(4, n // (y * z) // 4 * 4)
    if rng.random() < 0.4:      # extents that fit the blocks, and runs of eight of them along x
        x, y, z = max(64, x // 64 * 64), max(8, y // 8 * 8), max(4, z // 4 * 4) if dim == 3 else z
    return _draw_single(op, dim, mode, dtype, data, bound, x, y, z)


def _draw_single(*a):
    c = _single("", *a)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _count(case):
    return case["x"] if case["dim"] == 1 else case["x"] * case["y"] * case["z"]


def _field(n, seed, dtype, zero_runs):
    """Eight sinusoids over the index and N(0, 1e-3) noise; runs of 32..4096 values zeroed (20 %)."""
    r = np.random.default_rng(seed)
    f, a, ph = r.uniform(*FIELD_FREQ, 8), r.uniform(0.1, 1.0, 8), r.uniform(0, 2 * math.pi, 8)
    g = torch.Generator(device=DEV).manual_seed(seed)
    out = torch.empty(n, dtype=dtype, device=DEV)
    step = 1 << 26
    for s in range(0, n, step):
        m = min(step, n - s)
        i = torch.arange(s, s + m, dtype=torch.float64, device=DEV)
        v = torch.zeros(m, dtype=torch.float64, device=DEV)
        for k in range(8):
            v += torch.sin(i * (2 * math.pi * f[k]) + ph[k]) * a[k]
        v += torch.randn(m, dtype=torch.float32, device=DEV, generator=g) * 1e-3
        out[s:s + m] = v
    if zero_runs:
        k = max(1, int(0.2 * n / 2064))
        length = torch.from_numpy(r.integers(32, 4097, k)).to(DEV)
        start = torch.from_numpy((r.random(k) * n).astype(np.int64)).to(DEV)
        d = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
        one = torch.ones(k, dtype=torch.int32, device=DEV)
        d.index_add_(0, start, one)
        d.index_add_(0, (start + length).clamp_(max=n), -one)
        out[torch.cumsum(d, 0)[:n] > 0] = 0
    return out


def _grf(x, y, z, seed, dtype, spikes=1e-3):
    """A Gaussian random field of power spectrum k^-11/3 in [-50, 50], cut from the next powers of two
    (independent slices get a 2D field each in z by the same transform), with spikes of +-(100..1000)."""
    nx, ny, nz = (1 << max(3, (v - 1).bit_length()) for v in (x, y, z))
    nz = 1 if z == 1 else nz
    g = torch.Generator(device=DEV).manual_seed(seed)
    F = torch.fft.rfftn(torch.randn((nz, ny, nx), dtype=torch.float32, device=DEV, generator=g))
    k = (torch.fft.fftfreq(nz, device=DEV)[:, None, None] ** 2 + torch.fft.fftfreq(ny, device=DEV)[None, :, None] ** 2
         + torch.fft.rfftfreq(nx, device=DEV)[None, None, :] ** 2)
    k[0, 0, 0] = 1.0
    F *= k.pow_(-11.0 / 12.0)
    del k
    F[0, 0, 0] = 0
    v = torch.fft.irfftn(F, s=(nz, ny, nx), dim=(0, 1, 2))[:z, :y, :x].contiguous().reshape(-1)
    del F
    lo, hi = v.min(), v.max()
    v = (v - lo) / (hi - lo) * 100.0 - 50.0
    m = int(round(spikes * v.numel()))
    if m:                                        # one in each stretch of 1 / spikes values
        step = v.numel() // m
        at = torch.arange(m, device=DEV) * step + torch.randint(0, step, (m,), device=DEV, generator=g)
        u = torch.rand(m, device=DEV, generator=g) * 1800 - 900
        v[at] = u + 100 * torch.sign(u)
    return v.to(dtype).contiguous()


def _weight(n, seed, dtype, sigma=WEIGHT_SIGMA):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(n, dtype=torch.float32, device=DEV, generator=g) * sigma).to(dtype)


def _values(case, seed):
    n, t = _count(case), _dtype(case)
    if case["data"] == "grf":
        return _grf(case["x"], case["y"], case["z"], seed, t)
    if case["data"] == "weight":
        return _weight(n, seed, t)
    return _field(n, seed, t, zero_runs=n <= 1 << 27)


def _absolute(values, bound, data):
    """The absolute bound: as it is for weights, else relative to the value range, in float."""
    if data == "weight":
        return bound
    lo, hi = values.min().item(), values.max().item()
    if values.dtype == torch.float32:
        return float(np.float32(bound) * (np.float32(hi) - np.float32(lo)))
    return float(np.float32(bound) * np.float32(hi - lo))


def _batch_specs(case):
    """Sizes, types, modes and bounds of a batch's arrays: they belong to the case, the values to the seed."""
    r = np.random.default_rng(case["spec"])
    specs = []
    for i in range(case["count"]):
        n = int(round(math.exp(r.uniform(math.log(1024), math.log(case["largest"])))))
        f64 = bool(r.random() < 0.3)
        if i % 2 == 0:
            specs.append((n, f64, "fixed", "weight", 1e-3))
        else:
            specs.append((n, f64, "plain" if r.random() < 0.5 else "outlier", "field", float(r.choice([1e-2, 1e-3, 1e-4]))))
    return specs


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["op"].startswith("batch"):
        return _prepare_batch(case, seed)
    v = _values(case, seed)
    dims = (0, 0, 0) if case["dim"] == 1 else (case["x"], case["y"], case["z"])
    s = {"op": case["op"], "n": v.numel(), "dim": case["dim"], "dims": dims, "mode": P.MODES[case["mode"]],
         "type": 1 if case["dtype"] == "f64" else 0, "rel": case["bound"]}
    if s["op"] != "compress_rel":
        s["eb"] = _absolute(v, case["bound"], case["data"])
    s["cap"] = P.max_compressed_size(s["n"], s["dim"], dims, s["type"], s["mode"])
    stream = torch.zeros(s["cap"], dtype=torch.uint8, device=DEV)
    if s["op"] in ("compress", "compress_rel", "roundtrip"):
        s["values"], s["stream"] = v, stream
        if s["op"] == "roundtrip":
            s["out"] = torch.empty_like(v)
        return s
    size = P.compress_ex(v, stream, s["cap"], s["n"], s["eb"], s["dim"], dims, s["type"], s["mode"])
    s["size"] = size
    s["stream"] = stream[:size].clone()          # as read from a file
    s["out"] = torch.empty_like(v)
    if s["op"] == "report":
        P.decompress_ex(s["out"], s["stream"], s["n"], size, s["eb"], s["dim"], dims, s["type"], s["mode"])
        s["values"] = v
    return s


def _prepare_batch(case, seed):
    at, arrays = 0, []
    for i, (n, f64, mode, data, bound) in enumerate(_batch_specs(case)):
        t = torch.float64 if f64 else torch.float32
        k = seed * 1000 + i
        v = _weight(n, k, t) if data == "weight" else _field(n, k, t, True)
        cap = P.max_compressed_size(n, 1, (0, 0, 0), int(f64), P.MODES[mode])
        arrays.append({"values": v, "n": n, "eb": _absolute(v, bound, data), "type": int(f64), "mode": P.MODES[mode],
                       "cap": cap, "at": at})
        at += (cap + 255) // 256 * 256
    arena = torch.zeros(at, dtype=torch.uint8, device=DEV)       # every array's stream in one buffer
    q = torch.cuda.current_stream()
    items = [P.batch_item(a["values"], arena[a["at"]:], a["n"], a["cap"], a["eb"], 1, (0, 0, 0), a["type"], a["mode"])
             for a in arrays]
    s = {"op": case["op"], "arena": arena}
    if case["op"] == "batch_compress":
        s["values"] = [a["values"] for a in arrays]              # the plan holds their addresses
        s["plan"] = P.BatchPlan(items, P.BATCH_COMPRESS, graph=True, stream=q)
        return s
    with P.BatchPlan(items, P.BATCH_COMPRESS, stream=q) as plan:
        plan.execute(q)
        sizes, _ = plan.results(q)
    f32 = torch.zeros(sum((a["n"] + 63) // 64 * 64 for a in arrays if not a["type"]), dtype=torch.float32, device=DEV)
    f64 = torch.zeros(sum((a["n"] + 63) // 64 * 64 for a in arrays if a["type"]), dtype=torch.float64, device=DEV)
    used, items = [0, 0], []
    for a, size in zip(arrays, sizes):
        k = a["type"]
        items.append(P.batch_item(arena[a["at"]:], (f64 if k else f32)[used[k]:], a["n"], size, a["eb"], 1, (0, 0, 0), k, a["mode"]))
        used[k] += (a["n"] + 63) // 64 * 64
    s["out"] = [f32, f64]
    s["plan"] = P.BatchPlan(items, P.BATCH_DECOMPRESS, graph=True, stream=q)
    return s


def run(s):
    """One pass. A stream comes back as the whole buffer that it was written to (zeros after its end)."""
    op = s["op"]
    if op.startswith("batch"):
        q = torch.cuda.current_stream()
        s["plan"].execute(q)
        sizes, statuses = s["plan"].results(q)
        if op == "batch_compress":
            return s["arena"], np.array(sizes, dtype=np.int64), np.array(statuses, dtype=np.int64)
        return s["out"], np.array(statuses, dtype=np.int64)
    if op == "report":
        return P.quality(s["values"], s["out"]), P.ssim(s["values"], s["out"], s["dims"])
    shape = (s["dim"], s["dims"], s["type"], s["mode"])
    size = s.get("size")
    if op == "compress_rel":
        eb = P.rel_to_abs(s["values"], s["rel"])
        return s["stream"], P.compress_ex(s["values"], s["stream"], s["cap"], s["n"], eb, *shape), eb
    if op != "decompress":
        size = P.compress_ex(s["values"], s["stream"], s["cap"], s["n"], s["eb"], *shape)
        if op == "compress":
            return s["stream"], size
    P.decompress_ex(s["out"], s["stream"], s["n"], size, s["eb"], *shape)
    return s["out"] if op == "decompress" else (s["stream"], size, s["out"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its results in 64 bits
# ---------------------------------------------------------------------------
def _bytes(n, itemsize, data, mode, bound, op):
    values, stream = n * itemsize, n * STREAM_BYTES[(data, mode, bound)]
    if op == "report":
        return 2 * values
    if op == "roundtrip":
        return 2 * (values + stream)
    return values + stream                       # compress_rel too: the range and the stream from one read


def work(case):
    if case["op"].startswith("batch"):
        return {"bytes": sum(_bytes(n, 8 if f64 else 4, data, mode, bound, "")
                             for n, f64, mode, data, bound in _batch_specs(case)),
                "flops": 0}
    n = _count(case)
    flops = 0
    if case["op"] == "report" and min(case["x"], case["y"], case["z"]) >= 7:
        # sums over 7 x 7 x 7 windows moved by 2, axis by axis: five running sums
        flops = 5 * 7 * n
    return {"bytes": _bytes(n, 8 if case["dtype"] == "f64" else 4, case["data"], case["mode"], case["bound"], case["op"]),
            "flops": flops}


def _decoded(v, eb):
    """The values that the format's quantisation codes stand for, in 64 bits. The code of a value is defined by
    arithmetic in the value's type: t = x * (0.5 / eb), trunc(t + 0.5), less 1 where t < -0.5."""
    if v.dtype == torch.float32:
        r = float(np.float32(0.5) / np.float32(eb))
        eb = float(np.float32(eb))
    else:
        r = 0.5 / eb
    t = v * r
    q = torch.trunc(t + 0.5) - (t < -0.5).to(v.dtype)
    return q.double() * eb * 2


def exact(case, seed):
    op = case["op"]
    if op in ("compress", "batch_compress"):
        return None                              # bytes and lengths
    if op == "batch_decompress":
        out = [[], []]
        for i, (n, f64, _, data, bound) in enumerate(_batch_specs(case)):
            t, k = torch.float64 if f64 else torch.float32, seed * 1000 + i
            v = _weight(n, k, t) if data == "weight" else _field(n, k, t, True)
            d = _decoded(v, _absolute(v, bound, data))
            out[int(f64)] += [d, torch.zeros(-n % 64, dtype=torch.float64, device=DEV)]
        return [torch.cat(x) if x else torch.zeros(0, dtype=torch.float64, device=DEV) for x in out], None
    v = _values(case, seed)
    if op == "compress_rel":
        return None, None, case["bound"] * (v.max().double() - v.min().double()).item()
    d = _decoded(v, _absolute(v, case["bound"], case["data"]))
    if op == "decompress":
        return d
    if op == "roundtrip":
        return None, None, d
    d = d.to(v.dtype).double()
    return _quality(v.double(), d), _ssim(v.double(), d, case)


def _quality(o, d):
    n, e = o.numel(), (d - o).abs()
    mse, lo, hi = (e * e).mean().item(), o.min().item(), o.max().item()
    nz = o != 0
    a, b = o - o.mean(), d - d.mean()
    norm = math.sqrt(mse * n)
    return {"mse": mse, "range": hi - lo, "psnr": 20 * math.log10(hi - lo) - 10 * math.log10(mse), "norm_err": norm,
            "norm_err_norm": norm / math.sqrt((d * d).sum().item()), "nrmse": math.sqrt(mse) / (hi - lo),
            "max_abs_err": e.max().item(), "max_rel_err": (e[nz] / o[nz].abs()).max().item(),
            "correlation": ((a * b).mean() / (a * a).mean().sqrt() / (b * b).mean().sqrt()).item()}


def _ssim(o, d, case):
    """Mean over the 7 x 7 x 7 windows moved by 2 of luminance x contrast x structure."""
    shape = (case["z"], case["y"], case["x"])
    o, d = o.reshape(shape), d.reshape(shape)
    total, count = 0.0, 0
    for k in range(0, shape[0] - 6, 2):
        wx, wy = (v[k:k + 7].unfold(1, 7, 2).unfold(2, 7, 2).permute(1, 2, 0, 3, 4).flatten(2) for v in (o, d))
        mx, my = wx.mean(2), wy.mean(2)
        cx, cy = wx - mx[..., None], wy - my[..., None]
        vx, vy, vxy = (cx * cx).mean(2), (cy * cy).mean(2), (cx * cy).mean(2)
        r = wx.amax(2) - wx.amin(2)
        if case["dtype"] == "f32":
            r = r.float().double()
        r = torch.where(r == 0, torch.ones_like(r), r)
        c1, c2 = (0.01 * r) ** 2, (0.03 * r) ** 2
        sx, sy = vx.sqrt(), vy.sqrt()
        w = ((2 * mx * my + c1) / (mx * mx + my * my + c1) * (2 * sx * sy + c2) / (sx * sx + sy * sy + c2)
             * (vxy + c2 / 2) / (sx * sy + c2 / 2))
        total += w.sum().item()
        count += w.numel()
    return total / count
