"""Packed streams that end at every byte of a word and in chunks of every size
of their last word, in a buffer that ends with the archive: whole words go out
four at a time up to the stream's (or the buffer's) end, the rest byte by
byte, in the three-kernel and in the one-pass encode; archives must equal the
oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("chunks", [0, 1, 2, 9])
def test_last_words(gpu_ctx, chunks, fused):
    from vecsz_amd import VecszError, make_params

    ends = set()
    try:
        gpu_ctx.set_fused_encode(fused)
        for extra in range(1, 34):
            n = 1024 * chunks + 30 * extra + extra % 2
            r = np.random.default_rng(n)
            x = np.cumsum(r.integers(-9, 10, n)).astype(np.float32)
            ref, _, _ = po.compress(x, 0.5, False, 4096, 8)
            s = po.archive_sections(ref)
            ends.add((s["meta_bytes"] + s["huff_size"]) % 4)
            t = torch.from_numpy(x).cuda()
            out = torch.full((len(ref) + 64,), 0x5A, dtype=torch.uint8, device="cuda")
            p = make_params((n,), 0.5, "abs")
            size, _ = gpu_ctx.compress_into(p, t.data_ptr(), out.data_ptr(), len(ref))
            got = out.cpu().numpy()
            assert size == len(ref) and got[:size].tobytes() == ref and (got[size:] == 0x5A).all(), (n, fused)
            with pytest.raises(VecszError):
                gpu_ctx.compress_into(p, t.data_ptr(), out.data_ptr(), len(ref) - 1)
            assert (out.cpu().numpy()[size:] == 0x5A).all()
    finally:
        gpu_ctx.set_fused_encode(False)
    assert ends == {0, 1, 2, 3}
