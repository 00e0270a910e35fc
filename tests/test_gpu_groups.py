"""Batches beyond the Infinity Cache: their clusters are stepped in groups one
after the other within a call. The states are those of all clusters stepped
together (stream groups, the persistent kernel) bit for bit, at even and odd step
counts, and a NaN in any group halts the whole batch at its step."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from betse_amd.exceptions import BetseSimUnstableException
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def worlds():
    return batched_worlds(n_clusters=90, cells_range=(3800, 5000), grid_range=(100, 128), seed=11)


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
def test_groups_are_bit_identical(worlds, flux_mode):
    runs = []
    for tuning in (None, {"streams": 2}, {"exchange_form": 1}):
        say(f"case: {sum(c.n_cells for _, c in worlds)} cells, {flux_mode}, tuning {tuning}")
        b = batch(worlds, flux_mode, tuning=tuning)
        for n in (1, 2, 37):
            b.step_n(n)
        runs.append(state(b))
        b.close()
    for r in runs[1:]:
        for k in runs[0]:
            assert np.array_equal(runs[0][k], r[k]), k


@pytest.mark.parametrize("cluster", [0, 89])
def test_nan_halts_every_group(worlds, cluster):
    say(f"case: NaN in cluster {cluster}")
    b = batch(worlds, "fp64")
    b.step_n(6)
    b._dev["c_cell"][1, int(b.offsets[0][cluster]) + 3] = float("nan")
    with pytest.raises(BetseSimUnstableException) as e:
        b.step_n(34)
    assert e.value.step == 6
    before = state_raw(b)
    with pytest.raises(BetseSimUnstableException) as e:
        b.step_n(4)                       # (an odd count copies the workspace state back, halted or not)
    assert e.value.step == 6
    for k, v in state_raw(b).items():
        assert np.array_equal(v, before[k], equal_nan=True), k
    b.close()


def state_raw(b):
    b.stream.synchronize()
    return {k: b._dev[k].cpu().numpy().copy() for k in ("c_cell", "vm_cell", "c_env")}
