"""Uploads and downloads of a batch on both sides of the size from which they
go through pinned slots: what comes back is what went up, bit for bit."""
import numpy as np
import pytest

swe = pytest.importorskip("swe_ppm_amd")

pytestmark = pytest.mark.gpu


# fields of 4 MiB (copied straight both ways), 22 MiB in uneven blocks (downloads
# through the slots, which are used again, with a last piece of a few bytes) and
# just over 64 MiB (uploads too)
@pytest.mark.parametrize("sizes", [[(1022, 1022)], [(1500, 901), (62, 63), (1, 1), (2047, 2200)], [(4096, 4096)]])
def test_round_trip(sizes):
    rng = np.random.default_rng(len(sizes))
    blocks = [dict(nx=nx, ny=ny, bnd=[0, 1, 0, 1]) for nx, ny in sizes]
    with swe.SweBatch(blocks, solver=swe.AUGRIE, dx=1.0, dy=1.0) as batch:
        total = int(batch.sizes.sum())
        sent = [rng.random(total, dtype=np.float32) + 1.0 for _ in range(4)]
        batch.upload(*sent)
        back = batch.download(with_b=True, packed=True)
        for a, b in zip(sent, back):  # an upload sets the ghost cells only
            for u, v in zip(batch.unpack(a), batch.unpack(b)):
                assert np.array_equal(u[1:-1, 1:-1], v[1:-1, 1:-1])
        batch.upload(*back)
        for a, b in zip(back, batch.download(packed=True)):
            assert np.array_equal(a, b)
