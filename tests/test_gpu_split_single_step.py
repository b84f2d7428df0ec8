"""One step of flavour S through swe_hip_run costs what its three calls cost."""
import statistics
import time

import pytest

pytestmark = pytest.mark.gpu


# The device loop's start and end (time and dt to and from the GPU, three slots to
# clear) take 50 us that a single step does not win back: 84 to 92 us through the
# loop against 31 through the calls.
def test_single_step_costs_what_its_calls_cost(swe):
    from swe_ppm_amd import scenarios

    def median(f, count=60):
        times = []
        for _ in range(count):
            t0 = time.perf_counter()
            f()
            times.append(time.perf_counter() - t0)
        return statistics.median(times)

    with swe.SweBlock(64, 50, 15.0, 15.0, solver=swe.HLLE, flavour=swe.FLAVOUR_S) as blk:
        blk.set_boundaries([0] * 4)
        blk.init_seeded(scenarios.dam_break_islands_spec(5))

        def calls():
            blk.apply_bc()
            blk.update(blk.fluxes())
            blk.synchronize()

        blk.run(1), calls()
        assert median(lambda: blk.run(1)) < 1.6 * median(calls)
