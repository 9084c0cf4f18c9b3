"""A launch shape set by the caller is kept to, also one that names the defaults (engine.hip, shape_set):
only the automatic shape, or one that the autotuner chose, takes one block of 1024 threads per CU."""
import numpy as np
import pytest

from psim_amd import configs

pytestmark = pytest.mark.gpu

# 181 recorded steps of 40 sensors: windows of 3 flight caps (180 steps) in a CU's whole LDS, of one cap
# (60 steps) in a 256-thread block's share
WIDE, NARROW = 2, 4


def _start():
    import psim_amd
    cfg = configs.linear_bar(num_sensors=40, length=2000.0, num_phonons=400_000, num_measurements=181, sim_time=0.724,
                             spec=0.3, sim_type=1, step_interval=10).to_dict()
    engine = psim_amd.Engine(0)
    engine.set_tally_mode("lds")
    model = psim_amd.Model(cfg)
    model.upload(engine, 0)
    return engine, model


def _eager(engine, model, seed):
    engine.run_resident(seed)
    launches = engine.last_timing()["step_launches"]
    return engine.fetch(model.num_sensors, model.num_record), launches


def _same(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    assert a[2] == b[2]
    # FP64 sums of the same terms in another order: at most ~1e5 terms a tally
    assert np.allclose(a[1], b[1], rtol=0, atol=1e-11 * np.abs(b[1]).max())


@pytest.mark.parametrize("setter,value", [("set_grid", 8), ("set_grid", 3), ("set_block", 256), ("set_block", 512)])
def test_a_named_shape_is_kept_to(setter, value):
    engine, model = _start()
    ref, launches = _eager(engine, model, 4)
    assert launches == WIDE
    for seed in (4, 5):  # the graph of the automatic shape
        graph = engine.run_graph(model.num_sensors, model.num_record, seed)
    getattr(engine, setter)(value)
    res, launches = _eager(engine, model, 4)
    assert launches == NARROW
    _same(res, ref)
    again = engine.run_graph(model.num_sensors, model.num_record, 5)  # another sequence: captured again
    assert engine.last_timing()["step_launches"] == NARROW
    _same(again, graph)
    engine.set_window(0)  # automatic windows, of the named blocks
    assert _eager(engine, model, 4)[1] == NARROW
    engine.close()


@pytest.mark.parametrize("named", [False, True])
def test_the_autotuner_may_choose_the_automatic_shape(named):
    engine, model = _start()
    if named:
        engine.set_block(256)
    choice = engine.autotune(seed=1)
    print("autotune choice", choice, flush=True)
    automatic = (choice["window"], choice["blocks_per_cu"], choice["block"]) == (0, 8, 256)
    assert _eager(engine, model, 4)[1] == (WIDE if automatic else NARROW)
    engine.close()
