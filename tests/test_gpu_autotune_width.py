"""The autotuner on blocks that take the one-pass step: every width that it
reports a time for has run, and the one that it keeps runs afterwards."""
import pytest

pytestmark = pytest.mark.gpu


# A wave's columns are a chain: on 1024^2 cells 17 strips x 32 segments of 32
# columns leave the GPU's 1024 SIMDs half empty, and a launch of them takes more
# than twice one of 8 columns (59 against 23 us).
@pytest.mark.parametrize("solver", [0, 1])
def test_autotune_runs_the_widths_it_times(swe, solver):
    from swe_ppm_amd import scenarios

    n = 1024
    with swe.SweBlock(n, n, 1000.0 / n, 1000.0 / n, solver=solver) as blk:
        blk.set_boundaries([0] * 4)
        blk.init_seeded(scenarios.dam_break_islands_spec(5))
        ms = blk.autotune(100)
        assert ms[32] > 1.5 * ms[8], ms
        assert blk.get_tuning()[1] != 32
