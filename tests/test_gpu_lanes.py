"""Small runs spread over more waves of fewer lanes (engine.hip, SPREAD_WAVES_PER_CU): any phonon
count around the edges of that rule gives the oracle's run, on both tally paths."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phonons,blocks_per_cu", [(1, 8), (63, 8), (4097, 8), (9000, 1), (70001, 8), (70001, 1)])
@pytest.mark.parametrize("mode", ["lds", "hbm"])
def test_spread_runs_equal_the_oracle(phonons, blocks_per_cu, mode):
    import oracle
    import psim_amd
    cfg = configs.linear_bar(num_phonons=phonons, num_measurements=120, sim_time=0.6, spec=0.4).to_dict()
    ref = oracle.Model(cfg).run(9, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_grid(blocks_per_cu)
    engine.set_tally_mode(mode)
    model = psim_amd.Model(cfg)
    model.run(engine, 9)
    res = model.results(0)
    step, cause, xy = engine.fetch_fate(model.budget()[1])
    assert res.counters == ref.counters
    assert np.array_equal(step, ref.fate_step) and np.array_equal(cause, ref.fate_cause)
    assert np.array_equal(xy, ref.fate_xy) and np.array_equal(res.counts, ref.counts)
    # FP64 sums of the same terms in another order: at most ~1e4 terms a tally
    assert np.allclose(res.raw_flux, ref.flux, rtol=0, atol=1e-11 * max(1.0, np.abs(ref.flux).max()))
    engine.close()
