"""Flavour S's device loop (one launch per step) against its per-call API
(boundary conditions, fluxes, update), bit for bit: state with ghost cells, time,
every dt, and what a further per-call step makes of it."""
import numpy as np
import pytest

swe = pytest.importorskip("swe_ppm_amd")

pytestmark = pytest.mark.gpu


def _block(nx, ny, solver, bnd, seed):
    rng = np.random.default_rng(seed)
    shape = (nx + 2, ny + 2)
    b = rng.uniform(-0.5, 0.5, shape).astype(np.float32)
    h = rng.uniform(0.8, 2.0, shape).astype(np.float32)
    dry = rng.random(shape) < 0.03
    h[dry] = 0.0
    hu, hv = (np.where(dry, 0, rng.uniform(-0.3, 0.3, shape)).astype(np.float32) for _ in range(2))
    block = swe.SweBlock(nx, ny, 1.0, 1.5, solver=solver, flavour=swe.FLAVOUR_S)
    block.set_boundaries(bnd)
    block.upload(h, hu, hv, b)
    return block


# every strip width (1, 2, 4, 8, 16 columns and their remainders), strips of one
# row to three; walls, open sides and ghost cells that stay as they are (PASSIVE)
@pytest.mark.parametrize("xseg", [0, 4, 8, 16])
@pytest.mark.parametrize("nx,ny", [(1, 1), (7, 61), (33, 62), (130, 63), (41, 150)])
@pytest.mark.parametrize("solver", [swe.HLLE, swe.FWAVE, swe.AUGRIE, swe.HYBRID])
def test_loop_equals_per_call(solver, nx, ny, xseg):
    bnd = [(0, 0, 0, 0), (1, 0, 1, 5), (5, 1, 5, 1)][(nx + solver) % 3]
    for steps in (1, 2, 5):
        with _block(nx, ny, solver, bnd, nx) as one, _block(nx, ny, solver, bnd, nx) as two:
            if xseg:
                one.set_tuning(xseg=xseg)
            t, dts = one.run(steps)
            want, tw = [], np.float32(0)
            for _ in range(steps):
                two.apply_bc()
                want.append(two.fluxes())
                two.update(want[-1])
                tw = np.float32(tw + np.float32(want[-1]))
            assert np.array_equal(np.asarray(dts, np.float32), np.asarray(want, np.float32), equal_nan=True)
            assert np.float32(t) == tw or (np.isnan(t) and np.isnan(tw))
            for k in range(2):
                for a, c in zip(one.download(), two.download()):
                    assert np.array_equal(a, c, equal_nan=True)
                for block in (one, two):  # and on from there
                    block.apply_bc()
                    block.update(block.fluxes())
