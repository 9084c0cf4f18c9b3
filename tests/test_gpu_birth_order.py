"""The birth sort and the HBM tallies' prefix sums at the edges of their rules: steps that just fit
the emission blocks' LDS counters and steps that do not, bursts born in few steps, recorded steps
around the width of a scan block."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu

CASES = {
    "steps_fit_lds": configs.linear_bar(num_phonons=3000, num_measurements=36864, sim_time=1.0).to_dict(),
    "steps_past_lds": configs.linear_bar(num_phonons=3000, num_measurements=36865, sim_time=1.0).to_dict(),
    "burst": configs.film_transient(70_001, 255, 0.255, burst_duration=0.02),
    "one_scan_width": configs.linear_bar(num_phonons=2000, num_measurements=256, sim_time=0.8, sim_type=1,
                                         step_interval=16).to_dict(),
    "past_a_scan_width": configs.linear_bar(num_phonons=2000, num_measurements=257, sim_time=0.8, sim_type=1,
                                            step_interval=16).to_dict(),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_births_and_prefix_sums_equal_the_oracle(name):
    import oracle
    import psim_amd
    cfg = CASES[name]
    ref = oracle.Model(cfg).run(6, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_tally_mode("hbm")
    model = psim_amd.Model(cfg)
    model.run(engine, 6)
    res = model.results(0)
    step, cause, xy = engine.fetch_fate(model.budget()[1])
    assert res.counters == ref.counters
    assert np.array_equal(step, ref.fate_step) and np.array_equal(cause, ref.fate_cause)
    assert np.array_equal(xy, ref.fate_xy) and np.array_equal(res.counts, ref.counts)
    # FP64 sums of the same terms in another order: at most ~1e5 terms a tally
    assert np.allclose(res.raw_flux, ref.flux, rtol=0, atol=1e-11 * max(1.0, np.abs(ref.flux).max()))
    engine.close()
