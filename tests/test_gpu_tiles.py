"""Dual-quantization tiles that stop inside their Lorenzo blocks and load rows
ahead: extents on each side of a tile's planes, rows and columns, in every
tile form (64-wide, 4-wide with vector and element loads, padded, batched),
with outliers; archives must equal the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _field(shape, seed):
    r = np.random.default_rng(seed)
    x = np.cumsum(r.normal(0, 0.05, shape), axis=-1).astype(np.float32)
    x[r.random(shape) < 0.01] *= 1000  # outliers
    return x


@pytest.mark.parametrize("block", [8, 16, 32, 64])
@pytest.mark.parametrize("nx", [66, 259, 260])
def test_planes_and_rows(gpu_ctx, block, nx):
    fields = [_field((nz, ny, nx), nz + ny) for nz, ny in
              [(1, 7), (2, 8), (3, 9), (block - 1, 1), (block, 17), (block + 1, block - 1), (2 * block + 3, block + 1)]]
    fields += [_field((ny, nx), ny) for ny in (1, 7, 8, 9, block - 1, block + 9)]
    ts = [torch.from_numpy(f).cuda() for f in fields]
    refs = []
    for f, t in zip(fields, ts):
        print("tile", f.shape, block, flush=True)
        ref, n_ref, _ = po.compress(f, 1e-3, False, 1024, block)
        refs.append(ref)
        a, n = gpu_ctx.compress(t, 1e-3, "abs", block, 1024)
        assert n == n_ref and a.cpu().numpy().tobytes() == ref, f.shape
        pad, _, _ = po.compress(f, 1e-3, False, 1024, block, "block", "avg", 0.0)
        a, _ = gpu_ctx.compress(t, 1e-3, "abs", block, 1024, pad_mode="block", pad_type="avg")
        assert a.cpu().numpy().tobytes() == pad, f.shape
    for f, (a, _), ref in zip(fields, gpu_ctx.compress_batch(ts, 1e-3, "abs", block, 1024), refs):
        assert a.cpu().numpy().tobytes() == ref, f.shape


# enough 4-wide tiles for whole blocks, for half blocks and for quarter blocks
@pytest.mark.parametrize("shape", [(96, 344, 260), (192, 352, 512), (200, 704, 512)])
def test_tile_counts(gpu_ctx, shape):
    x = _field(shape, 5)
    ref, n_ref, _ = po.compress(x, 1e-3, False, 4096, 8)
    a, n = gpu_ctx.compress(torch.from_numpy(x).cuda(), 1e-3, "abs")
    assert n == n_ref and a.cpu().numpy().tobytes() == ref
