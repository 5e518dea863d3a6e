"""Performance cases of the compression path: what a program that uses this
package has it do, called through `vecsz_amd.Context`.

A case is one call: compress or decompress of one field, decompress with the
decode index that was kept beside the archive, or a batch of fields in one
call.  Fields live on the GPU and stay there.  The data are those of the
benchmark: Gaussian random fields with a turbulence-like spectrum (`grf`),
sums of plane waves plus noise (`waves`), and random walks with spikes
(`walk`), see `vecsz_amd.datagen`.
"""
import math
import random

import numpy as np
import torch

from vecsz_amd import Context, datagen, make_params

#: Elements of the fields that `draw` gives: 64 KiB to 512 MiB of float32.
SMALLEST, LARGEST = 16 << 10, 1 << 27
#: Elements of one field of a batch, 64 KiB to 4 MiB of float32.
BATCH_SMALLEST, BATCH_LARGEST = 16 << 10, 1 << 20


def _case(op, data, shape, eb, mode, block=8, dict_size=4096, pad_mode="none", pad_type="const", fields=1, name=None):
    z, y, x = (0,) * (3 - len(shape)) + tuple(shape)
    c = {"op": op, "data": data, "z": z, "y": y, "x": x, "eb": eb, "mode": mode, "block": block,
         "dict_size": dict_size, "pad_mode": pad_mode, "pad_type": pad_type, "fields": fields}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # A simulation snapshot of 1 GiB: the benchmark's default field.
        _case("compress", "grf", (1024, 512, 512), 1e-4, "r2r", name="compress_3d_1gib"),
        _case("decompress", "grf", (1024, 512, 512), 1e-4, "r2r", name="decompress_3d_1gib"),
        # The same kind of field at 512^3 with a looser bound, decompressed by
        # a program that kept the decode index beside the archive.
        _case("decompress_indexed", "grf", (512, 512, 512), 1e-3, "r2r", name="decompress_indexed_3d_512"),
        # A field with no extent a multiple of anything, an absolute bound,
        # larger blocks, a smaller dictionary and per-block average padding.
        _case("compress", "grf", (201, 333, 413), 1e-2, "abs", 16, 1024, "block", "avg", name="compress_3d_padded"),
        # A climate-like 2D slice of 1800 x 3600, absolute bound.
        _case("compress", "waves", (1800, 3600), 1e-4, "abs", name="compress_2d_slice"),
        _case("decompress", "waves", (1800, 3600), 1e-4, "abs", name="decompress_2d_slice"),
        # A 256 MiB 1D stream (particle data, a sensor) with outliers.
        _case("compress", "walk", (1 << 26,), 1e-4, "r2r", name="compress_1d_stream"),
        _case("decompress", "walk", (1 << 26,), 1e-4, "r2r", name="decompress_1d_stream"),
        # The smallest field: a call is all latency and launches.
        _case("compress", "grf", (25, 25, 26), 1e-3, "r2r", name="compress_3d_small"),
        _case("decompress", "grf", (25, 25, 26), 1e-3, "r2r", name="decompress_3d_small"),
        # Many small ragged 2D and 3D fields in one call, as an AMR code or a
        # serving process has them.
        _case("compress_batch", "grf", (), 0.0, "r2r", fields=48, name="compress_batch_small"),
        _case("decompress_batch", "grf", (), 0.0, "r2r", fields=48, name="decompress_batch_small"),
    ]


def _shape(rng, ndim, n):
    """A shape of about n elements, its extents as they come (odd ones too)."""
    if ndim == 1:
        return (n,)
    if ndim == 2:
        y = max(8, int(math.sqrt(n) * math.exp(rng.uniform(-0.7, 0.7))))
        return (y, max(8, n // y))
    z = max(8, int(n ** (1 / 3) * math.exp(rng.uniform(-0.7, 0.4))))
    y = max(8, int(math.sqrt(n / z) * math.exp(rng.uniform(-0.4, 0.4))))
    return (z, y, max(8, n // (z * y)))


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    op = rng.choice(["compress", "compress", "decompress", "decompress", "decompress_indexed", "compress_batch",
                     "decompress_batch"])
    block = rng.choice([8, 8, 8, 16, 32, 64])
    dict_size = rng.choice([1024, 4096, 4096, 4096])
    if op.endswith("_batch"):
        return _case(op, "grf", (), 0.0, "r2r", block, dict_size, fields=rng.randint(16, 48))
    ndim = rng.choice([1, 2, 2, 3, 3, 3])
    data = {1: "walk", 2: rng.choice(["grf", "waves"]), 3: "grf"}[ndim]
    mode = rng.choice(["abs", "r2r"])
    # grf spans 100, waves about 8, a walk with its spikes about 2000
    eb = rng.choice([1e-4, 1e-3, 1e-2]) * (1 if mode == "r2r" else {"grf": 100, "waves": 1, "walk": 1000}[data])
    pad_mode = rng.choice(["none", "none", "none", "global", "block", "edge"])
    # (the global average is one sum in index order: too slow to be used on large fields)
    pad_type = rng.choice(["max", "min", "const"] if pad_mode == "global" else ["max", "min", "avg", "const"])
    dict_size = rng.choice([dict_size, dict_size, dict_size, 65536])
    return _case(op, data, _shape(rng, ndim, _log_uniform(rng, SMALLEST, LARGEST)), eb, mode, block, dict_size,
                 pad_mode, pad_type)


# ------------------------------------------------------------------ inputs


def _waves(shape, seed):
    """datagen.sinusoids_2d's field, evaluated on the GPU."""
    rng = random.Random(seed)
    y = torch.arange(shape[0], dtype=torch.float64, device="cuda")[:, None]
    x = torch.arange(shape[1], dtype=torch.float64, device="cuda")[None, :]
    f = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for _ in range(8):
        k = 2 * math.pi / rng.uniform(50.0, 900.0)
        amp, phase, theta = rng.uniform(0.0, 1.0), rng.uniform(0.0, 2 * math.pi), rng.uniform(0.0, 2 * math.pi)
        f += amp * torch.sin(math.cos(theta) * k * x + math.sin(theta) * k * y + phase)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    f += 1e-3 * torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
    return f.to(torch.float32)


def _fields(case, seed):
    """[(field, error bound)] of a case."""
    if case["op"].endswith("_batch"):
        # half 2D, half 3D, each with its own size and bound; the shapes are
        # the case's, the values the seed's
        rng = random.Random(case["fields"])
        out = []
        for k in range(case["fields"]):
            shape = _shape(rng, 2 + k % 2, _log_uniform(rng, BATCH_SMALLEST, BATCH_LARGEST))
            eb = rng.choice([1e-2, 1e-3, 1e-4])
            out.append((datagen.grf(shape, seed=1000 * seed + k, device="cuda", pow2=True), eb))
        return out
    shape = tuple(case[k] for k in "zyx" if case[k])
    if case["data"] == "walk":
        x = datagen.walk_spikes_1d(shape[0], seed=seed, device="cuda")
    elif case["data"] == "waves":
        x = _waves(shape, seed)
    else:
        x = datagen.grf(shape, seed=seed, device="cuda", pow2=True)
    return [(x, case["eb"])]


def _range(x):
    """max - min as the reference takes it, in float32."""
    return float((x.max() - x.min()).item())


def prepare(case, seed):
    fields = _fields(case, seed)
    ctx = Context(0)
    s = {"case": case, "ctx": ctx}
    how = {"block": case["block"], "dict_size": case["dict_size"]}
    pad = {"pad_mode": case["pad_mode"], "pad_type": case["pad_type"], "pad_constant": 0.5}
    if case["op"] == "compress":
        x = fields[0][0]
        p = make_params(tuple(reversed(x.shape)), case["eb"], case["mode"], **how, **pad)
        s["x"], s["args"] = x, dict(eb=case["eb"], mode=case["mode"], **how, **pad)
        s["out"] = torch.zeros(ctx.compress_bound(p), dtype=torch.uint8, device="cuda")
    elif case["op"] == "compress_batch":
        s["x"] = [f for f, _ in fields]
        s["params"] = [make_params(tuple(reversed(f.shape)), e, case["mode"], **how) for f, e in fields]
        s["out"] = [torch.zeros(ctx.compress_bound(p), dtype=torch.uint8, device="cuda") for p in s["params"]]
    elif case["op"] == "decompress_batch":
        got = ctx.compress_batch([f for f, _ in fields], [e for _, e in fields], case["mode"], **how)
        s["archives"] = [a.clone() for a, _ in got]
        s["args"] = dict(modes=case["mode"], value_ranges=[_range(f) for f, _ in fields], **how)
    else:
        x = fields[0][0]
        s["args"] = dict(mode=case["mode"], value_range=_range(x) if case["mode"] == "r2r" else 0.0, **how)
        if case["op"] == "decompress_indexed":
            a, _, s["args"]["index"] = ctx.compress_indexed(x, case["eb"], case["mode"], **how, **pad)
        else:
            a, _ = ctx.compress(x, case["eb"], case["mode"], **how, **pad)
        s["archive"] = a.clone()
    return s


def run(state):
    ctx, op = state["ctx"], state["case"]["op"]
    if op == "compress":
        archive, n_outlier = ctx.compress(state["x"], out=state["out"], **state["args"])
        return {"archive": state["out"], "bytes": archive.numel(), "n_outlier": n_outlier}
    if op == "compress_batch":
        out = state["out"]
        got = ctx.compress_batch_into(state["params"], [x.data_ptr() for x in state["x"]],
                                      [o.data_ptr() for o in out], [o.numel() for o in out])
        return {"archives": out, "sizes": np.array(got)}
    if op == "decompress_batch":
        return ctx.decompress_batch(state["archives"], **state["args"])
    return ctx.decompress(state["archive"], **state["args"])


# ------------------------------------------------------------------ what is needed, and what is exact


def _bits_per_value(data, eb):
    """Archive bits per value, about (eb relative to the field's range)."""
    if data == "walk":
        return 3.0
    return min(16.0, max(2.0, 2.7 + 3.2 * math.log10(1e-2 / eb)))


def work(case):
    """One read of the input and one write of the output: 4 bytes a value and
    the archive, whose size is that of typical data."""
    if case["op"].endswith("_batch"):
        rng = random.Random(case["fields"])
        total = 0.0
        for k in range(case["fields"]):
            shape = _shape(rng, 2 + k % 2, _log_uniform(rng, BATCH_SMALLEST, BATCH_LARGEST))
            total += math.prod(shape) * (4 + _bits_per_value("grf", rng.choice([1e-2, 1e-3, 1e-4])) / 8)
        return {"bytes": int(total), "flops": 0}
    n = math.prod(case[k] for k in "zyx" if case[k])
    span = {"grf": 100.0, "waves": 8.0, "walk": 2000.0}[case["data"]]
    eb = case["eb"] if case["mode"] == "r2r" else case["eb"] / span
    b = n * (4 + _bits_per_value(case["data"], eb) / 8)
    if case["op"] == "decompress_indexed":
        b += n / 128 * 6.25
    return {"bytes": int(b), "flops": 0}


def _quantized(x, eb, case):
    """The values an archive of x stands for: the multiple of 2 eb that the
    format's prequantization (a float32 product, to nearest; in the columns
    past the last whole group of eight of a 3D field, a float64 product, half
    away from zero) picks for each value, in 64 bits."""
    if case["mode"] == "r2r":
        eb = eb * _range(x)
    r = 1 / (2 * eb)
    q = torch.round(x * torch.tensor(r, dtype=torch.float32)).to(torch.float64)
    tail = x.shape[-1] // 8 * 8
    if x.dim() == 3 and tail < x.shape[-1]:
        p = x[..., tail:].to(torch.float64) * r
        q[..., tail:] = torch.sign(p) * torch.floor(p.abs() + 0.5)
    elif x.dim() == 2:
        q[..., tail:] = 0  # the reference codes no values there
    return q * (2 * eb)


def exact(case, seed):
    # archives are bytes; a 1D block predicted from a raw pad value is not a
    # multiple of the step
    if not case["op"].startswith("decompress") or (case["data"] == "walk" and case["pad_mode"] != "none"):
        return None
    got = [_quantized(x, eb, case) for x, eb in _fields(case, seed)]
    return got if case["op"] == "decompress_batch" else got[0]
