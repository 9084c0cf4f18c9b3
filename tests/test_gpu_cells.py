"""Both forms in which the transport kernel reads a cell (engine_device.hpp, Tri and Edge): a model whose
edges all have few sub-surfaces runs on Tri, one with an edge of more than TRI_SUB_BITS count on Edge."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu


def comb(teeth: int, sim_type: int) -> dict:
    """A strip under `teeth` narrow cells, hot on the left and cold on the right."""
    b = configs.ModelBuilder(60, 0.3, 20_000, 300.0, sim_type, 10 if sim_type else 0)
    strip, top = b.add_sensor(300.0), b.add_sensor(300.0)
    b.add_rectangle((0, 0), (2.0 * teeth, 20), strip, 0.4)
    for i in range(teeth):
        b.add_rectangle((2.0 * i, 20), (2.0 * i + 2, 30), top, 0.4)
    b.add_surface((0, 0), (0, 20), 310.0)
    b.add_surface((2.0 * teeth, 0), (2.0 * teeth, 20), 290.0)
    return b.to_dict()


# sub-surfaces of the strip's upper edge: the most a Tri holds, one more
@pytest.mark.parametrize("teeth", [15, 16])
@pytest.mark.parametrize("sim_type,mode", [(0, "hbm"), (1, "hbm"), (1, "lds")])
def test_cells_equal_the_oracle(teeth, sim_type, mode):
    import oracle
    import psim_amd
    cfg = comb(teeth, sim_type)
    ref = oracle.Model(cfg).run(8, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_tally_mode(mode)
    model = psim_amd.Model(cfg)
    for precision, block, rel in (("fp64", 256, 1e-11), ("fp64", 512, 1e-11), ("fp32_kahan", 256, 1e-4)):
        engine.set_tally_precision(precision)
        engine.set_block(block)
        model.run(engine, 8)
        res = model.results(0)
        step, cause, xy = engine.fetch_fate(model.budget()[1])
        assert res.counters == ref.counters
        assert np.array_equal(step, ref.fate_step) and np.array_equal(cause, ref.fate_cause)
        assert np.array_equal(xy, ref.fate_xy) and np.array_equal(res.counts, ref.counts)
        # sums of the same terms in another order: at most ~1e4 terms a tally, each rounded to 2^-53 (2^-24)
        assert np.allclose(res.raw_flux, ref.flux, rtol=0, atol=rel * max(1.0, np.abs(ref.flux).max()))
    engine.close()


# sensors alike (one record in scalar registers) and not (one of them starts at another temperature)
@pytest.mark.parametrize("mode", ["hbm", "lds"])
@pytest.mark.parametrize("alike", [True, False])
def test_sensors_equal_the_oracle(alike, mode):
    import oracle
    import psim_amd
    cfg = configs.linear_bar(num_sensors=5, num_phonons=20_000, num_measurements=100, sim_time=0.5, spec=0.5, sim_type=1,
                             step_interval=10).to_dict()
    if not alike:
        cfg["sensors"][3]["t_init"] = 302.0
    ref = oracle.Model(cfg).run(5, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    engine.set_tally_mode(mode)
    model = psim_amd.Model(cfg)
    model.run(engine, 5)
    res = model.results(0)
    for got, want in zip(engine.fetch_fate(model.budget()[1]), (ref.fate_step, ref.fate_cause, ref.fate_xy)):
        assert np.array_equal(got, want)
    assert res.counters == ref.counters and np.array_equal(res.counts, ref.counts)
    # FP64 sums of the same terms in another order: at most ~1e4 terms a tally
    assert np.allclose(res.raw_flux, ref.flux, rtol=0, atol=1e-11 * max(1.0, np.abs(ref.flux).max()))
    engine.close()


# one block of 1024 threads per CU from 1024 phonons per CU on (engine.hip, RunPlan::wide_free), tables in
# LDS; in full simulations each bin's rates too, with impurities and without
@pytest.mark.parametrize("short,t_eq,impurities", [(1, 300.0, True), (0, 300.0, True), (1, 0.0, True), (0, 0.0, True),
                                                   (0, 0.0, False)])
def test_wide_untallied_blocks_equal_the_oracle(short, t_eq, impurities):
    import oracle
    import psim_amd
    total = 1024 * 256 - 2 * short  # an MI355X has 256 CUs
    cfg = configs.linear_bar(num_phonons=total, num_measurements=60, sim_time=0.12, spec=0.5, t_eq=t_eq).to_dict()
    if not impurities:
        for m in cfg["materials"]:
            m["r_data"]["b_i"] = 0.0
    ref = oracle.Model(cfg).run(5, nthreads=8, fate=True)
    engine = psim_amd.Engine(0)
    engine.set_fate(True)
    model = psim_amd.Model(cfg)
    model.run(engine, 5)
    res = model.results(0)
    assert abs(model.budget()[1] - total) <= 1
    for got, want in zip(engine.fetch_fate(model.budget()[1]), (ref.fate_step, ref.fate_cause, ref.fate_xy)):
        assert np.array_equal(got, want)
    assert res.counters == ref.counters and np.array_equal(res.counts, ref.counts)
    engine.close()
