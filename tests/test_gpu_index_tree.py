"""Decompress with a decode index of an archive whose tree is damaged: refused,
with nothing written, whatever an earlier call left in the context."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(4099,), (70, 130), (9, 20, 70), (12, 40, 300)])
def test_damaged_tree(gpu_ctx, shape):
    from vecsz_amd import VecszError, datagen

    x = torch.from_numpy(datagen.grf(shape, seed=len(shape)).astype(np.float32)).cuda()
    a, _, idx = gpu_ctx.compress_indexed(x, 1e-3, "abs")
    raw = bytearray(a.cpu().numpy().tobytes())
    nd = len(shape)
    pad = int(np.frombuffer(bytes(raw[4 * nd + 12: 4 * nd + 20]), np.uint64)[0])
    h = 4 * nd + 36 + 4 * pad
    nodes = int.from_bytes(raw[h: h + 4], "big")
    assert nodes > 1
    w = 1 if nodes <= 256 else 2
    raw[h + 9: h + 9 + w] = b"\xff" * w if w == 2 else b"\x00"  # the root's left child: no node of the tree
    bad = torch.from_numpy(np.frombuffer(bytes(raw), np.uint8).copy()).cuda()
    gpu_ctx.decompress(a, "abs", index=idx)  # (leaves codes in the context)
    out = torch.full(shape, -7.25, device="cuda")
    with pytest.raises(VecszError):
        gpu_ctx.decompress(bad, "abs", index=idx, out=out)
    assert bool((out == -7.25).all())
    with pytest.raises(VecszError):
        gpu_ctx.decompress(bad, "abs", out=out)
    assert bool((out == -7.25).all())
