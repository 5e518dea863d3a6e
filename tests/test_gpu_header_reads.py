"""Decompress reads an archive's headers in one round trip: behind a pad
section, and with the tree where the host builds the tables (dictionaries over
4096); a second one only for what lies past the first read."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# 9^3 pad values, none, and 35,937 of them (past the first read)
@pytest.mark.parametrize("shape, pad, dict_size, index, waits", [
    ((64, 64, 64), "block", 4096, False, 1),
    ((64, 64, 64), "block", 4096, True, 1),
    ((64, 64, 64), "block", 65536, False, 1),
    ((64, 64, 64), "none", 65536, False, 1),
    ((64, 64, 64), "none", 65536, True, 1),
    ((60, 62, 61), "none", 4096, False, 1),
    ((256, 256, 256), "block", 4096, False, 2),
])
def test_round_trips(gpu_ctx, shape, pad, dict_size, index, waits):
    from vecsz_amd import datagen

    x = datagen.grf(shape, seed=7).astype(np.float32)
    how = dict(pad_mode=pad, pad_type="avg") if pad != "none" else {}
    xt = torch.from_numpy(x).cuda()
    if index:
        a, _, idx = gpu_ctx.compress_indexed(xt, 1e-2, "abs", 8, dict_size, **how)
    else:
        a, idx = gpu_ctx.compress(xt, 1e-2, "abs", 8, dict_size, **how)[0], None
    gpu_ctx.enable_timing(True)
    try:
        y = gpu_ctx.decompress(a, "abs", 0.0, 8, dict_size, index=idx)
        names = [n for n, _ in gpu_ctx.timings()]
    finally:
        gpu_ctx.enable_timing(False)
    assert names.count("header") == waits
    ref = po.decompress(a.cpu().numpy().tobytes(), x.shape, False, 0.0, dict_size, 8)
    assert np.array_equal(y.cpu().numpy().reshape(-1).view(np.uint32), np.asarray(ref).reshape(-1).view(np.uint32))
