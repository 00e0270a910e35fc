"""What the steps run with is what running_tuning reports: the persistent kernel on
small problems, the exchange in the env kernel on larger ones, the forced variants
once any are forced; forcing what is reported changes nothing."""

import numpy as np
import pytest

import bench
from betse_amd.batch import batched_worlds
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu

SMALL = dict(n_clusters=3, cells_range=(30, 200), grid_range=(16, 24))
FUSED = dict(n_clusters=4, cells_range=(1800, 2400), grid_range=(48, 64))      # more than 512 cell tiles
FORCED = {"mem_waves": 1, "env_ions_per_block": 2, "exchange_form": 1, "persistent": 0, "streams": 2}


@pytest.mark.parametrize("size,want", [(SMALL, dict(persistent=1)),
                                       (FUSED, dict(persistent=0, exchange_form=2, env_ions_per_block=5))])
def test_running_tuning(size, want):
    say(f"case: {size}")
    worlds = batched_worlds(seed=13, **size)
    b = batch(worlds, "fp64")
    run = b.running_tuning()
    assert {k: run[k] for k in want} == want and run["serial_groups"] == 1
    b.step_n(23)
    ref = state(b)
    names = bench.step_kernel_names(run, False)
    assert names == (("step_team",) if run["persistent"] else ("mem_cell", "env_field_exchange"))
    b.close()
    b = batch(worlds, "fp64", tuning={k: v for k, v in run.items() if k != "serial_groups"})
    assert b.running_tuning() == run
    b.step_n(23)
    for k, v in state(b).items():
        assert np.array_equal(v, ref[k]), k
    b.set_tuning(FORCED)
    assert {k: b.running_tuning()[k] for k in FORCED} == FORCED
    b.close()


def test_kernels_are_timed_as_the_steps_run_them():
    """With the exchange in the env kernel there is no exchange launch to time."""
    b = batch(batched_worlds(seed=13, **FUSED), "fp64")
    env, ex = b.time_kernel("env_field_exchange", 20), b.time_kernel("env_exchange", 20)
    say(f"case: kernels of fused steps, env {env * 1e3:.1f} us, exchange {ex * 1e3:.1f} us")
    assert ex < 0.2 * env
    b.close()


def test_without_graphs_every_kernel_is_a_launch():
    """use_graph = 0 on a small problem: separate launches, with the same bits."""
    worlds = batched_worlds(seed=13, **SMALL)
    states = []
    for use_graph in (True, False):
        b = batch(worlds, "fp64")
        b.use_graph = use_graph
        say(f"case: use_graph {use_graph}, running {b.running_tuning()}")
        assert b.running_tuning()["persistent"] == int(use_graph)
        b.step_n(23)
        states.append(state(b))
        b.set_tuning({"persistent": 1})
        assert b.running_tuning()["persistent"] == 1
        b.close()
    for k, v in states[0].items():
        assert np.array_equal(v, states[1][k]), k
