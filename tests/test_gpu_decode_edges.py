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


def _sections(a):
    """(archive bytes, offset of the Huffman section, its size, outlier count)."""
    nd = int(np.frombuffer(a[:4], np.int32)[0])
    pad, huff, nout = (int(v) for v in np.frombuffer(a[4 * nd + 12: 4 * nd + 36], np.uint64))
    return 4 * nd + 36 + 4 * pad, huff, nout


def _renumbered(a, seed):
    """The archive with its tree's nodes (but the root) in another order."""
    h, huff, _ = _sections(a)
    nc = int.from_bytes(a[h: h + 4], "big")
    w = 1 if nc <= 256 else 2
    ty = np.uint8 if w == 1 else np.uint16
    t = h + 9
    left, right = (np.frombuffer(a[t + i * nc * w: t + (i + 1) * nc * w], ty).astype(np.int64) for i in (0, 1))
    sym = np.frombuffer(a[t + 2 * nc * w: t + 2 * nc * w + 4 * nc], np.uint32)
    leaf = np.frombuffer(a[t + 2 * nc * w + 4 * nc: t + 2 * nc * w + 5 * nc], np.uint8)
    to = np.concatenate([[0], 1 + np.random.default_rng(seed).permutation(nc - 1)])
    out = [np.empty(nc, ty), np.empty(nc, ty), np.empty(nc, np.uint32), np.empty(nc, np.uint8)]
    out[0][to] = np.where(left > 0, to[left], 0)
    out[1][to] = np.where(right > 0, to[right], 0)
    out[2][to], out[3][to] = sym, leaf
    return a[:t] + b"".join(o.tobytes() for o in out) + a[t + nc * (2 * w + 5):]


# trees whose nodes are not numbered parents first: the host builds their
# tables (the device leaves them), alone, with an index and in a batch
@pytest.mark.parametrize("nsym", [40, 900])
def test_other_node_orders(gpu_ctx, nsym):
    counts = [1 + (i * i) % 37 for i in range(nsym)]
    x = _field(counts, seed=nsym)
    xt = torch.from_numpy(x).cuda()
    a, _, idx = gpu_ctx.compress_indexed(xt, 0.5, "abs")
    ref = gpu_ctx.decompress(a, "abs")
    b = torch.from_numpy(np.frombuffer(_renumbered(a.cpu().numpy().tobytes(), nsym), np.uint8).copy()).cuda()
    assert not torch.equal(a, b)
    for y in [gpu_ctx.decompress(b, "abs"), gpu_ctx.decompress(b, "abs", index=idx),
              *gpu_ctx.decompress_batch([a, b, a], "abs")]:
        assert torch.equal(y.view(torch.int32), ref.view(torch.int32))


# a stream that is a byte short is refused, also where the codewords that a
# table entry holds at once would reach past its end
@pytest.mark.parametrize("tail", [0, 5, 64, 600])
def test_short_stream(gpu_ctx, tail):
    from vecsz_amd import VecszError

    x = np.concatenate([_field([3] * 64 + [2000], seed=tail), np.zeros(tail, np.float32)])
    a, _ = gpu_ctx.compress(torch.from_numpy(x).cuda(), 0.5, "abs")
    raw = a.cpu().numpy().tobytes()
    h, huff, nout = _sections(raw)
    nd = int(np.frombuffer(raw[:4], np.int32)[0])
    cut = raw[: 4 * nd + 20] + np.uint64(huff - 1).tobytes() + raw[4 * nd + 28: h + huff - 1] + raw[h + huff:]
    c = torch.from_numpy(np.frombuffer(cut, np.uint8).copy()).cuda()
    with pytest.raises(VecszError):
        gpu_ctx.decompress(c, "abs")
    with pytest.raises(VecszError):
        gpu_ctx.decompress_batch([a, c], "abs")
