"""Batches beyond the Infinity Cache, whose clusters are stepped in groups one after
the other: in two groups and in more, the states are those of separate launches over
the whole batch, bit for bit."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def worlds():
    return batched_worlds(n_clusters=90, cells_range=(3800, 5000), grid_range=(100, 128), seed=11)


@pytest.mark.parametrize("flux_mode,copies,groups", [("fp64", 1, 2), ("fp64", 2, 3), ("fp32", 2, 3)])
def test_groups_are_the_whole_batch(worlds, flux_mode, copies, groups):
    runs = []
    for use_graph in (True, False):
        b = batch(worlds * copies, flux_mode)
        b.use_graph = use_graph
        n_groups = b.running_tuning()["serial_groups"]
        say(f"case: {b.n_cells} cells, {flux_mode}, graphs {use_graph}, {n_groups} groups")
        assert n_groups == (groups if use_graph else 1)
        for n in (16, 21):
            b.step_n(n)
        runs.append(state(b))
        b.close()
    for k in runs[0]:
        assert np.array_equal(runs[0][k], runs[1][k]), k


def test_the_split_does_not_depend_on_the_order_of_the_clusters(worlds):
    """A cluster in which fewer ions move, first and last, in a batch of just over 2.2
    times the cache."""
    p, cells = worlds[0]
    p = p.copy()
    p.mem_perms = dict(p.mem_perms, Cl=0.0)
    rest = (worlds * 2)[1:]
    groups = []
    for w in ([(p, cells)] + rest, rest + [(p, cells)]):
        b = batch(w, "fp32")
        groups.append(b.running_tuning()["serial_groups"])
        say(f"case: a cluster without Cl flux at {'the start' if w[0][0] is p else 'the end'}: {groups[-1]} groups")
        b.close()
    assert groups == [3, 3]
