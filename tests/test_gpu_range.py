"""States at the edges of the range in which the sweeps use their short
divisions and square roots (dev::in_normal_range in solvers_dev.hpp): a wave
with a cell outside it runs its tile in the general form.  Both forms round
correctly, so every state is bit-identical to the oracle."""
import numpy as np
import pytest

from helpers import same_bits

pytestmark = pytest.mark.gpu

KINDS = ["fast", "deep", "tiny", "vacuum", "near_dry"]


def _state(kind, nx=70, ny=131, seed=5):
    """Random water with cells of one kind strewn over it."""
    rng = np.random.default_rng(seed)
    shape = (nx + 2, ny + 2)
    h = rng.uniform(0.5, 10.0, shape)
    u, v = rng.uniform(-2.0, 2.0, (2, *shape))
    b = rng.uniform(-1.0, 1.0, shape)
    h[rng.random(shape) < 0.05] = 0.0
    some = rng.random(shape) < 0.02
    pick = lambda *values: rng.choice(np.array(values), size=int(some.sum()))  # noqa: E731
    if kind == "fast":  # velocities around 2^20
        u[some] = pick(2.0**20, -(2.0**20), 2.0**20 - 1, 2.0**20 + 1, 2.0**19, 2.0**21)
        v[some] = pick(0.0, 1.0, 2.0**19)
    elif kind == "deep":  # depth and bed around 2^40
        h[some] = pick(2.0**39, 2.0**40, 2.0**41)
        b[some] = pick(0.0, 2.0**39, -(2.0**40))
    elif kind == "tiny":  # momenta down to denormal numbers and signed zeros
        scale = 10.0 ** rng.uniform(-45.0, -20.0, shape)
        u, v = u * scale, v * scale
        h[:] = np.where(rng.random(shape) < 0.5, 4.0, h)
        b[:] = np.where(rng.random(shape) < 0.5, 0.0, b)
        u[some] = pick(0.0, -0.0)
    elif kind == "vacuum":  # strong expansions: a middle state of zero depth
        u = np.where(rng.random(shape) < 0.5, 40.0, -40.0)
    f = [a.astype(np.float32) for a in (h, h * u, h * v, b)]
    if kind == "near_dry":  # depths at the dry tolerance and the clamp
        dry = np.float32(0.01)
        f[0][some] = pick(dry, np.nextafter(dry, np.float32(0)), np.nextafter(dry, np.float32(1)), 1e-30, 0.1)
    return f


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("solver", [0, 1, 2, 3])
def test_range_edges_bitwise(swe, oracle, solver, kind):
    state, bnd = _state(kind), [0, 1, 0, 1]
    nx, ny = state[0].shape[0] - 2, state[0].shape[1] - 2
    ref = oracle.run_u(*state, 2.0, 3.0, bnd, solver, 2)
    assert all(np.isfinite(a).all() for a in ref)
    for strategy in (0, 1, 2):
        with swe.SweBlock(nx, ny, 2.0, 3.0, solver=solver) as blk:
            blk.set_boundaries(bnd)
            blk.set_tuning(strategy, -1)
            blk.upload(*state)
            _, dts = blk.run(2)
            got = (*blk.download(), dts)
        for name, a, c in zip(("h", "hu", "hv", "dt"), got, ref):
            assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]) if a.ndim == 2 else same_bits(a, c), (strategy, name)
    block = dict(nx=nx, ny=ny, dx=2.0, dy=3.0, bnd=bnd)
    for fused in (0, 1):
        with swe.SweBatch([block], solver=solver) as bt:
            bt.set_tuning(fused=fused)
            bt.upload(*[[a] for a in state])
            bt.run(2)
            got = [a[0] for a in bt.download()]
        for name, a, c in zip(("h", "hu", "hv"), got, ref):
            assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), ("batch", fused, name)
    ref = oracle.run_s(*state, 2.0, bnd, solver, 1)
    with swe.SweBlock(nx, ny, 2.0, 2.0, solver=solver, flavour=swe.FLAVOUR_S) as blk:
        blk.set_boundaries(bnd)
        blk.upload(*state)
        blk.run(1)
        got = blk.download()
    for name, a, c in zip(("h", "hu", "hv"), got, ref):
        assert same_bits(a[1:-1, 1:-1], c[1:-1, 1:-1]), ("split", name)
