"""Wide recording windows (engine.hip, wide_window_for) of models whose sensors differ and of batches: the
kernels that read a sensor's record for each phonon, against the oracle."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu


def _bar(sensors, phonons, steps, sim_time):
    cfg = configs.linear_bar(num_sensors=sensors, length=50.0 * sensors, num_phonons=phonons, num_measurements=steps,
                             sim_time=sim_time, spec=0.3, sim_type=1, step_interval=10).to_dict()
    cfg["sensors"][sensors // 2]["t_init"] = 303.0
    return cfg


def _compare(res, ref):
    np.testing.assert_array_equal(res.counts, ref.counts)
    # FP64 sums of the same terms in another order: at most ~1e5 terms a tally
    assert np.allclose(res.raw_flux, ref.flux, rtol=0, atol=1e-11 * max(1.0, np.abs(ref.flux).max()))


# windows of 3 flight caps of 60 steps: one window's last step, one past it
@pytest.mark.parametrize("steps,launches", [(180, 1), (181, 2)])
def test_unlike_sensors_in_wide_windows(steps, launches):
    import oracle
    import psim_amd
    cfg = _bar(40, 300_000, steps, 0.002 * steps)
    ref = oracle.Model(cfg).run(7, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_tally_mode("lds")
    model = psim_amd.Model(cfg)
    model.run(engine, 7)
    assert engine.last_timing()["step_launches"] == launches
    res = model.results(0)
    for got, want in zip(engine.fetch_fate(model.budget()[1]), (ref.fate_step, ref.fate_cause, ref.fate_xy)):
        np.testing.assert_array_equal(got, want)
    assert res.counters == ref.counters
    _compare(res, ref)
    engine.close()


# 15 sensors each: a cap of 128 steps, which a CU's LDS holds twice for 30 sensors (256 steps a window)
@pytest.mark.parametrize("steps,launches", [(256, 1), (300, 2)])
def test_batches_in_wide_windows(steps, launches):
    import oracle
    import psim_amd
    cfgs = [_bar(15, 150_000 + 7 * i, steps, 0.002 * steps) for i in range(2)]
    cfgs[1]["sensors"][0]["t_init"] = 296.0
    engine = psim_amd.Engine(0)
    engine.set_tally_mode("lds")
    models = [psim_amd.Model(c) for c in cfgs]
    counters = psim_amd.run_batch(engine, models, seed=7)
    assert engine.last_timing()["step_launches"] == launches
    summed = {k: 0 for k in counters}
    for i, (cfg, model) in enumerate(zip(cfgs, models)):
        single = oracle.Model(cfg)
        single.set_stream(i)
        ref = single.run(7, nthreads=8)
        _compare(model.results(0), ref)
        for k, v in ref.counters.items():
            summed[k] += v
    assert counters == summed
    engine.close()
