"""Streams in which one codeword repeats over thousands of subsequences: a
constant, masked or very smooth stretch of a field, where a table entry holds
several codewords and the subsequences' decodes reach one another's ends in
other steps.  They must settle without waiting for one another (each stage
"decode_redo" beyond the first is a host check and its passes), and the fields
must equal the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _field(d):
    """The 1D field whose quant codes (B 8, abs eb 0.5) are the deltas d."""
    n = d.size
    return np.concatenate([d, np.zeros(-n % 8, d.dtype)]).reshape(-1, 8).cumsum(axis=1).reshape(-1)[:n].astype(np.float32)


def _checks(ctx, f):
    """f()'s result, and the redo stages it took."""
    ctx.enable_timing(True)
    try:
        y = f()
        return y, sum(n == "decode_redo" for n, _ in ctx.timings())
    finally:
        ctx.enable_timing(False)


def _check(ctx, x, eb, r2r, most, most_batch):
    print("runs", x.shape, flush=True)
    vr = po.value_range(x) if r2r else 0.0
    a, _, _ = po.compress(x, eb, r2r, 4096, 8)
    ref = po.decompress(a, x.shape, r2r, vr, 4096, 8).reshape(-1).view(np.uint32)
    at = torch.from_numpy(np.frombuffer(a, np.uint8).copy()).cuda()
    mode = "r2r" if r2r else "abs"
    y, redo = _checks(ctx, lambda: ctx.decompress(at, mode, vr))
    assert np.array_equal(y.cpu().numpy().reshape(-1).view(np.uint32), ref)
    ys, redo_batch = _checks(ctx, lambda: ctx.decompress_batch([at, at.clone()], mode, vr))
    for y in ys:
        assert np.array_equal(y.cpu().numpy().reshape(-1).view(np.uint32), ref)
    assert redo <= most and redo_batch <= most_batch, (redo, redo_batch)


# The bounds: passes that a list needs where a start is right as soon as it is
# on the codewords of the one before it (counted for these streams one
# codeword at a time), in the launches' batches of passes.


# a run of one 2-bit codeword, which every start inside it finds, and noise of
# 17 codewords behind it
@pytest.mark.parametrize("run", [1 << 17, 1 << 21])
def test_run_in_step(gpu_ctx, run):
    noise = np.random.default_rng(run).integers(-8, 9, run)
    _check(gpu_ctx, _field(np.concatenate([np.zeros(run + 3, noise.dtype), noise])), 0.5, False, 1, 1)


# noise and runs by turns; a run that begins on an odd bit is a chain of all
# its subsequences (256 and 1,024: more than one workgroup's rounds)
@pytest.mark.parametrize("run, count, most_batch", [(1 << 16, 40, 19), (1 << 18, 6, 64)])
def test_runs_in_noise(gpu_ctx, run, count, most_batch):
    rng = np.random.default_rng(run)
    noise = rng.integers(-8, 9, (count, 20000))
    d = [np.concatenate([q, np.zeros(run + int(rng.integers(0, 9)), q.dtype)]) for q in noise]
    _check(gpu_ctx, _field(np.concatenate(d)), 0.5, False, 2, most_batch)


# one 2-bit codeword with 1 in 100 and 1 in 3,000 others
@pytest.mark.parametrize("others, most_batch", [(100, 2), (3000, 9)])
def test_rare_others(gpu_ctx, others, most_batch):
    n = (1 << 21) + 3
    rng = np.random.default_rng(others)
    d = np.where(rng.random(n) * others < 1, rng.integers(-8, 9, n), 0)
    _check(gpu_ctx, _field(d), 0.5, False, 1, most_batch)


# 4 and 16 symbols of equal count: 2 and 3 to 5 bits, an entry holds 6 and 2
# to 4, and 512 bits are no whole number of entries
@pytest.mark.parametrize("symbols", [4, 16])
def test_equal_counts(gpu_ctx, symbols):
    d = np.repeat(np.arange(symbols) - symbols // 2, (1 << 20) // symbols)
    np.random.default_rng(symbols.bit_length() - 1).shuffle(d)
    _check(gpu_ctx, _field(d), 0.5, False, 1, 1)


# a 3D field of which nine tenths are masked (codewords of 2 to 19 bits)
def test_masked_field(gpu_ctx):
    from vecsz_amd import datagen

    x = datagen.grf((32, 160, 192), seed=5)
    x = np.where(x < np.quantile(x, 0.9), 0, x).astype(np.float32)
    _check(gpu_ctx, x, 1e-3, True, 1, 5)


# streams of 21,721 and 77,592 subsequences whose first pass leaves a list
# that one workgroup takes (964 and 106 entries): one host check
@pytest.mark.parametrize("data", ["walk", "grf"])
def test_short_list_of_a_long_stream(gpu_ctx, data):
    from vecsz_amd import datagen

    x = datagen.walk_spikes_1d(1 << 22) if data == "walk" else datagen.grf((64, 256, 256), seed=3)
    _check(gpu_ctx, x.astype(np.float32), 1e-4, True, 1, 5)
