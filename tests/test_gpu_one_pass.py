"""The one-pass step of the light solvers (kernels_advance.hpp), which the
device loop takes on blocks of 2^19 cells and more: shapes at the edges of its
61-row strips and its column segments, every kind of side."""
import numpy as np
import pytest

from helpers import same_bits

pytestmark = pytest.mark.gpu

SHAPES = [(8600, 61), (8460, 62), (4300, 122), (4265, 123), (33, 15900), (9, 58300), (1, 524288), (725, 731)]


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("solver", [0, 1])
def test_one_pass_matches_oracle_and_store_strategy(swe, oracle, solver, nx, ny):
    rng = np.random.default_rng(nx + ny)
    shape = (nx + 2, ny + 2)
    h = rng.uniform(0.2, 5.0, shape).astype(np.float32)
    h[rng.random(shape) < 0.1] = 0.0
    hu, hv = [(h * rng.uniform(-2.0, 2.0, shape)).astype(np.float32) for _ in range(2)]
    b = rng.uniform(-1.0, 1.0, shape).astype(np.float32)
    state = (h, hu, hv, b)
    for bnd, widths in (([0, 1, 0, 1], (-1, 8)), ([1, 0, 1, 0], (16, 32)), ([5, 0, 3, 1], (-1,))):
        got = {}
        for strategy, width in [(1, -1)] + [(2, w) for w in widths]:
            with swe.SweBlock(nx, ny, 1.0, 1.5, solver=solver) as blk:
                blk.set_boundaries(bnd)
                blk.set_tuning(strategy, width)
                blk.upload(*state)
                t1, d1 = blk.run(1)
                t2, d2 = blk.run(2, t1)
                got[strategy, width] = (*blk.download(), np.concatenate([d1, d2]), np.array([t2], np.float32))
        for key, out in got.items():  # ghosts included
            for name, a, c in zip(("h", "hu", "hv", "dt", "t"), out, got[1, -1]):
                assert same_bits(a, c), (bnd, key, name)
        if max(bnd) <= 1:  # the oracle's loop sets every ghost cell
            ref = oracle.run_u(*state, 1.0, 1.5, bnd, solver, 3)
            for name, a, c in zip(("h", "hu", "hv"), got[2, widths[0]], ref):
                assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), (bnd, name)
            assert same_bits(got[2, widths[0]][3], ref[3])


# Hybrid takes it from 6 Mi cells on, with both kinds of edge among the cells
@pytest.mark.parametrize("nx,ny", [(103200, 61), (31, 203000), (2510, 2511)])
def test_one_pass_hybrid_matches_oracle_and_store_strategy(swe, oracle, nx, ny):
    rng = np.random.default_rng(nx)
    shape = (nx + 2, ny + 2)
    h = rng.uniform(0.5, 4.0, shape).astype(np.float32)
    h[rng.random(shape) < 0.02] = 0.0
    hu, hv = [(h * rng.uniform(-2.0, 2.0, shape)).astype(np.float32) for _ in range(2)]
    state, bnd = (h, hu, hv, rng.uniform(-0.5, 0.5, shape).astype(np.float32)), [1, 0, 0, 1]
    got = {}
    for strategy, width in ((1, -1), (2, -1), (2, 16)):
        with swe.SweBlock(nx, ny, 1.0, 1.5, solver=3) as blk:
            blk.set_boundaries(bnd)
            blk.set_tuning(strategy, width)
            blk.upload(*state)
            _, dts = blk.run(3)
            got[strategy, width] = (*blk.download(), dts)
    for key, out in got.items():  # ghosts included
        for name, a, c in zip(("h", "hu", "hv", "dt"), out, got[1, -1]):
            assert same_bits(a, c), (key, name)
    ref = oracle.run_u(*state, 1.0, 1.5, bnd, 3, 3)
    for name, a, c in zip(("h", "hu", "hv"), got[2, -1], ref):
        assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), name
    assert same_bits(got[2, -1][3], ref[3])
