"""Flavour S on a block of more columns than the second dimension of a launch
grid (65536) holds at four per workgroup: loop and calls against the oracle."""
import numpy as np
import pytest

from helpers import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [4 * 32768 - 2, 4 * 32768 - 1, 4 * 65535 - 2, 4 * 65535 - 1, 600_001])
def test_wide_block(swe, oracle, nx):
    ny, steps, bnd = 3, 2, [0, 1, 0, 0]
    rng = np.random.default_rng(nx)
    shape = (nx + 2, ny + 2)
    h = rng.uniform(1.0, 3.0, shape).astype(np.float32)
    hu, hv = (rng.uniform(-0.3, 0.3, shape).astype(np.float32) for _ in range(2))
    b = rng.uniform(-0.5, 0.5, shape).astype(np.float32)
    ref = oracle.run_s(h, hu, hv, b, 2.0, bnd, swe.FWAVE, steps)
    with swe.SweBlock(nx, ny, 2.0, 2.0, solver=swe.FWAVE, flavour=swe.FLAVOUR_S) as blk:
        blk.set_boundaries(bnd)
        for loop in (True, False):
            blk.upload(h, hu, hv, b)
            if loop:
                _, dts = blk.run(steps)
            else:
                dts = []
                for _ in range(steps):
                    blk.apply_bc()
                    dts.append(blk.fluxes())
                    blk.update(dts[-1])
            for a, c in zip(blk.download(), ref):
                assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), loop
            assert same_bits(np.asarray(dts, np.float32), ref[3]), loop
