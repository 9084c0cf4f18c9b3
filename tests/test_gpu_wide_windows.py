"""Wide recording windows (engine.hip, wide_window_for): several flight caps per launch in a CU's
whole LDS give the run of the narrow windows, which an explicit block size asks for."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu


# sensors, recorded steps, launches of wide windows: caps 128, 60, 23 -> windows of 15, 3, 3 caps;
# ends on a window's edge and one step past it; 60 sensors' cap of 39 fits three times (117)
@pytest.mark.parametrize("sensors,steps,launches", [(4, 300, 1), (40, 180, 1), (40, 181, 2), (60, 300, 3), (100, 140, 3)])
def test_wide_windows_equal_narrow_ones(sensors, steps, launches):
    import psim_amd
    cfg = configs.linear_bar(num_sensors=sensors, length=50.0 * sensors, num_phonons=400_000, num_measurements=steps,
                             sim_time=0.004 * steps, spec=0.3, sim_type=1, step_interval=10).to_dict()
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_tally_mode("lds")
    model = psim_amd.Model(cfg)

    def run():
        model.run(engine, 4)
        return model.results(0), engine.fetch_fate(model.budget()[1]), engine.last_timing()["step_launches"]

    wide, wide_fate, n = run()
    assert n == launches
    engine.set_block(128)
    narrow, narrow_fate, _ = run()
    assert wide.counters == narrow.counters
    assert np.array_equal(wide.counts, narrow.counts)
    for a, b in zip(wide_fate, narrow_fate):
        assert np.array_equal(a, b)
    # FP64 sums of the same terms in another order: at most ~1e5 terms a tally
    assert np.allclose(wide.raw_flux, narrow.raw_flux, rtol=0, atol=1e-11 * np.abs(narrow.raw_flux).max())
    engine.close()
