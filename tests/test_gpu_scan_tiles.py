"""The scan of chunk bits and outliers: fields whose chunks end on each side of
a tile's 4096, and of the most one workgroup scans (four tiles), alone and as a
batch that crosses tiles inside its fields; archives must equal the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CHUNK = 1024


def _field(n, seed):
    r = np.random.default_rng(seed)
    x = np.cumsum(r.integers(-3, 4, n)).astype(np.float32)
    x[:: 5 * CHUNK + 3] += 1e5  # outliers all along
    return x


@pytest.mark.parametrize("chunks", [4095, 4096, 4097, 3 * 4096, 4 * 4096 - 1, 4 * 4096, 4 * 4096 + 1, 5 * 4096 + 7])
def test_tiles(gpu_ctx, chunks):
    n = chunks * CHUNK - 5
    print("scan", chunks, flush=True)
    x = _field(n, chunks)
    t = torch.from_numpy(x).cuda()
    ref, n_ref, _ = po.compress(x, 0.5, False, 1024, 8)
    a, got = gpu_ctx.compress(t, 0.5, "abs", 8, 1024)
    assert got == n_ref and a.cpu().numpy().tobytes() == ref


def test_batch_over_tiles(gpu_ctx):
    fs = [_field(c * CHUNK + 1, c) for c in (5, 4090, 3, 6000, 4096, 4100, 1)]
    got = gpu_ctx.compress_batch([torch.from_numpy(f).cuda() for f in fs], 0.5, "abs", 8, 1024)
    for f, (a, _) in zip(fs, got):
        assert a.cpu().numpy().tobytes() == po.compress(f, 0.5, False, 1024, 8)[0], f.shape
