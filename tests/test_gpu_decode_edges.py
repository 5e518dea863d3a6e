"""The Huffman decoders where their units end: streams of a chosen number of
subsequences (one, one less and one more than a sync or write workgroup's),
streams whose codewords never synchronise, and code lengths on each side of
what a table level, a window and a pair of codewords hold.  Single, indexed
and batched decodes must equal the oracle's output bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _field(counts, seed=0, dict_size=4096):
    """A 1D field whose quant codes (B 8, abs eb 0.5) are the deltas
    -len/2 .. len/2 with the given counts, shuffled."""
    k = len(counts)
    d = np.repeat(np.arange(k) - k // 2, counts)
    np.random.default_rng(seed).shuffle(d)
    n = d.size
    pad = -n % 8
    q = np.concatenate([d, np.zeros(pad, d.dtype)]).reshape(-1, 8).cumsum(axis=1).reshape(-1)[:n]
    assert np.abs(q).max(initial=0) < 1 << 21 and k <= dict_size
    return q.astype(np.float32)


def _check(ctx, x, dict_size=4096, index=True):
    print("decode", x.size, dict_size, flush=True)
    a_ref, _, _ = po.compress(x, 0.5, False, dict_size, 8)
    y_ref = po.decompress(a_ref, x.shape, False, 0.0, dict_size, 8).reshape(-1).view(np.uint32)
    xt = torch.from_numpy(x).cuda()
    a, _, idx = ctx.compress_indexed(xt, 0.5, "abs", 8, dict_size)
    assert a.cpu().numpy().tobytes() == a_ref
    y = ctx.decompress(a, "abs", 0.0, 8, dict_size)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), y_ref)
    y = ctx.decompress(a, "abs", 0.0, 8, dict_size, index=idx)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), y_ref)
    if dict_size <= 4096:
        for y in ctx.decompress_batch([a, a[: a.numel()].clone(), a], "abs", 0.0, 8, dict_size):
            assert np.array_equal(y.cpu().numpy().view(np.uint32), y_ref)


# 256 symbols of equal count: 8-bit codewords, 64 to a subsequence of 512 bits
@pytest.mark.parametrize("nsub", [1, 2, 510, 511, 512, 513, 1022, 1023, 1024, 1025])
@pytest.mark.parametrize("extra", [0, 1])
def test_subsequence_counts(gpu_ctx, nsub, extra):
    n = 64 * nsub + extra
    _check(gpu_ctx, _field([n // 256 + (i < n % 256) for i in range(256)] if n >= 256 else [1] * n, seed=nsub))


# 32 symbols of equal count: 5-bit codewords, which a decode from a wrong bit
# never leaves, so every subsequence waits for the one before it
@pytest.mark.parametrize("nsub", [3, 40])
def test_never_synchronises(gpu_ctx, nsub):
    n = 512 * nsub // 5 // 32 * 32
    _check(gpu_ctx, _field([n // 32] * 32, seed=nsub))


# counts that double (or grow as the Fibonacci numbers): one codeword of each
# length up to 19 (28), past the first level's 12 bits, the second's 16 and
# the pair's window; dict 65536 with its symbols past 4095 takes the 32-bit
# tables
@pytest.mark.parametrize("dict_size", [4096, 65536])
@pytest.mark.parametrize("growth", ["double", "fibonacci"])
def test_code_lengths(gpu_ctx, dict_size, growth):
    counts = [1, 1]
    while len(counts) < (20 if growth == "double" else 29):
        counts.append(2 * counts[-1] if growth == "double" else counts[-1] + counts[-2])
    _check(gpu_ctx, _field(counts, seed=len(counts)), dict_size)


# thousands of rare symbols beside common ones: more second-level tables than
# a workgroup keeps in LDS
@pytest.mark.parametrize("common", [4, 64])
def test_many_long_codewords(gpu_ctx, common):
    counts = [1 + i % 3 for i in range(3900)]
    counts[1950 - common // 2: 1950 + common // 2] = [4000] * common
    _check(gpu_ctx, _field(counts, seed=common))
