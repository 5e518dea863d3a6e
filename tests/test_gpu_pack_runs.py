"""Bit packing in runs of chunks with codewords joined by fours: run lengths of
1 to 8 chunks and their ends, chunks where two neighbouring codewords do not
fit one word, codewords over 26 and over 32 bits, every codebook form, and the
index; archives must equal the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CHUNK = 1024


@pytest.fixture
def ctx():
    from vecsz_amd import Context

    return Context(0)


def _skewed(n, seed, levels=24):
    """Steps whose counts are Fibonacci numbers (the deepest Huffman tree for
    their sum), the rarest side by side."""
    r = np.random.default_rng(seed)
    fib = [1, 1]
    while len(fib) < levels and sum(fib) + fib[-1] + fib[-2] <= n // 2:
        fib.append(fib[-1] + fib[-2])
    d = np.repeat(np.arange(len(fib)), fib[::-1])
    d = np.concatenate([np.zeros(n - len(d), np.int64), d])
    k = n - 64
    head = r.permutation(d[:k])  # the last 64, the rarest, stay together
    at = int(r.integers(0, k))
    d = np.concatenate([head[:at], d[k:], head[at:]])
    s = np.where(r.random(n) < 0.5, -1, 1)
    return np.cumsum(d * s).astype(np.float32)


def _check(ctx, x, eb, dict_size, index=True):
    t = torch.from_numpy(x).cuda()
    ref, n_ref, _ = po.compress(x, eb, False, dict_size, 8)
    a, n = ctx.compress(t, eb, "abs", 8, dict_size)
    assert n == n_ref and a.cpu().numpy().tobytes() == ref, x.shape
    if index:
        b, _, idx = ctx.compress_indexed(t, eb, "abs", 8, dict_size)
        assert b.cpu().numpy().tobytes() == ref, x.shape
        full = ctx.decompress(a, "abs", 0.0, 8, dict_size)
        assert torch.equal(ctx.decompress(b, "abs", 0.0, 8, dict_size, index=idx), full)


# one workgroup: runs of 1 (under 16 chunks), 2 (16 on), 4 (32 on) and 8 (64 on)
@pytest.mark.parametrize("chunks", [1, 3, 4, 5, 15, 16, 17, 31, 33, 63, 64, 65, 97])
@pytest.mark.parametrize("grid", [1, 2048])
def test_runs(ctx, chunks, grid):
    ctx.set_launch_shape(768, grid)
    for extra in (-1, 0, 1, 17):
        n = chunks * CHUNK + extra
        print("run", chunks, extra, grid, flush=True)
        r = np.random.default_rng(n)
        x = np.cumsum(r.normal(0, 3, n)).astype(np.float32)
        x[r.random(n) < 0.003] += 1e5  # outliers, here and there
        _check(ctx, x, 0.5, 1024)


@pytest.mark.parametrize("dict_size", [64, 1024, 4096, 16384])
def test_deep_codewords(ctx, dict_size):
    for n, grid in ((50_001, 1), (400_003, 2), (400_003, 2048)):
        print("deep", n, dict_size, grid, flush=True)
        ctx.set_launch_shape(768, grid)
        _check(ctx, _skewed(n, n), 0.5, dict_size)


def test_deep_batch(ctx):
    fs = [_skewed(n, n) for n in (1023, 30_000, 260_001)] + [_skewed(4096 * 40, 3).reshape(64, 2560)]
    refs = [po.compress(f, 0.5, False, 4096, 8)[0] for f in fs]
    for grid in (1, 3, 2048):
        ctx.set_launch_shape(768, grid)
        got = ctx.compress_batch([torch.from_numpy(f).cuda() for f in fs], 0.5, "abs")
        for f, ref, (a, _) in zip(fs, refs, got):
            assert a.cpu().numpy().tobytes() == ref, (f.shape, grid)
