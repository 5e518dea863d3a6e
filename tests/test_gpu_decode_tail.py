"""Streams whose subsequences find their codewords late (a walk of short
codewords, long chains of wrong starts): the short lists that one workgroup
resolves and the long ones that it leaves, in both table forms; the fields must
equal the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# lists of a few, of some hundreds and, after the first passes, of thousands
@pytest.mark.parametrize("n", [1 << 18, (1 << 22) + 5, 1 << 25])
@pytest.mark.parametrize("dict_size", [4096, 65536])
def test_chains(gpu_ctx, n, dict_size):
    from vecsz_amd import datagen

    x = datagen.walk_spikes_1d(n).astype(np.float32)
    vr = po.value_range(x)
    print("tail", n, dict_size, flush=True)
    ref, _, _ = po.compress(x, 1e-4, True, dict_size, 8)
    a = torch.from_numpy(np.frombuffer(ref, np.uint8).copy()).cuda()
    y = gpu_ctx.decompress(a, "r2r", vr, 8, dict_size).cpu().numpy()
    yo = po.decompress(ref, x.shape, True, vr, dict_size, 8)
    assert np.array_equal(y.view(np.uint32).ravel(), np.asarray(yo).view(np.uint32).ravel())


# 8-bit codewords, 64 to a subsequence of 512 bits, 512 of those to a write
# unit: on each side of the 64 units whose offsets one workgroup finds
@pytest.mark.parametrize("nsub", [511 * 64, 512 * 63 + 1, 512 * 64 - 1, 512 * 64, 512 * 64 + 1])
def test_units(gpu_ctx, nsub):
    n = 64 * nsub
    d = np.arange(n) % 256 - 128
    np.random.default_rng(nsub).shuffle(d)
    x = d.reshape(-1, 8).cumsum(axis=1).reshape(-1).astype(np.float32)
    print("units", nsub, flush=True)
    ref, _, _ = po.compress(x, 0.5, False, 4096, 8)
    a = torch.from_numpy(np.frombuffer(ref, np.uint8).copy()).cuda()
    y = gpu_ctx.decompress(a, "abs", 0.0, 8, 4096).cpu().numpy()
    assert np.array_equal(y.ravel(), x)
