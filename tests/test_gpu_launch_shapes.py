"""Launch shapes on each side of the packer's own limit (1024 workgroups, half
of the shape above it): the same archive, with every run of chunks in place."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# 9000 chunks: more than four to a workgroup at each shape
def test_encode_shapes():
    from vecsz_amd import Context

    ctx = Context(0)
    n = 9000 * 1024 + 77
    x = np.cumsum(np.random.default_rng(3).integers(-9, 10, n)).astype(np.float32)
    ref, _, _ = po.compress(x, 0.5, False, 4096, 8)
    t = torch.from_numpy(x).cuda()
    for grid in (1, 1000, 1024, 1025, 2047, 2048, 2049, 2051, 4096, 65536):
        print("shape", grid, flush=True)
        ctx.set_launch_shape(768, grid)
        a, _ = ctx.compress(t, 0.5, "abs")
        assert a.cpu().numpy().tobytes() == ref, grid
