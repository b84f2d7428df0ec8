"""Small blocks run strips of 1, 2, 4 or 8 columns (narrow_width in swe_hip.hip)
until the caller sets a width: the device loop and the per-call loop at the
edges of the strips, and across the sizes where the width changes."""
import numpy as np
import pytest

from helpers import same_bits

pytestmark = pytest.mark.gpu

# 1 column, then 2 and 4 columns for some solvers (see narrow_width's limits)
SHAPES = [(1, 1), (2, 63), (3, 62), (5, 125), (33, 61), (300, 190), (700, 130), (1300, 250)]


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("solver", [0, 1, 2, 3])
def test_narrow_strips_match_oracle(swe, oracle, solver, nx, ny):
    rng = np.random.default_rng(7 * nx + ny)
    shape = (nx + 2, ny + 2)
    h = rng.uniform(0.2, 5.0, shape).astype(np.float32)
    h[rng.random(shape) < 0.1] = 0.0
    still = rng.random(shape) < 0.5
    hu, hv = [np.where(still, 0, h * rng.uniform(-2.0, 2.0, shape)).astype(np.float32) for _ in range(2)]
    b = np.where(still, 0, rng.uniform(-1.0, 1.0, shape)).astype(np.float32)
    state, bnd, steps = (h, hu, hv, b), [0, 1, 1, 0], 5
    ref = oracle.run_u(*state, 1.0, 1.5, bnd, solver, steps)
    with swe.SweBlock(nx, ny, 1.0, 1.5, solver=solver) as blk:
        blk.set_boundaries(bnd)
        blk.upload(*state)
        _, dts = blk.run(steps)
        loop = (*blk.download(), dts)
        blk.upload(*state)
        dts = []
        for _ in range(steps):
            blk.apply_bc()
            dts.append(blk.fluxes())
            blk.update(dts[-1])
        calls = (*blk.download(), np.array(dts, np.float32))
    for got in (loop, calls):
        for name, a, c in zip(("h", "hu", "hv"), got, ref):
            assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), name
        assert same_bits(got[3], ref[3])
