"""decompress_batch of archives held as signed and unsigned bytes: their
headers are read as bytes whatever the type."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_mixed_byte_types(gpu_ctx):
    x = [torch.randn(40, 50 + k, device="cuda") for k in range(3)]
    a = [gpu_ctx.compress(t, 1e-2, "abs")[0] for t in x]
    want = gpu_ctx.decompress_batch(a, "abs")
    for k, y in enumerate(gpu_ctx.decompress_batch([a[0], a[1].view(torch.int8), a[2]], "abs")):
        assert y.shape == x[k].shape and torch.equal(y, want[k])
