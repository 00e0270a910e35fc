"""After a NaN every cluster of a batch is at the step that produced the first of
them, whichever way the steps ran: with NaNs that come up at different steps in
different clusters, the state, the gates and the fields are those of separate
launches of the three kernels over the whole batch, bit for bit."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from betse_amd.channels import draw_channel_state
from betse_amd.exceptions import BetseSimUnstableException
from tests.test_gpu_configs import batch, say

pytestmark = pytest.mark.gpu

SEPARATE = {"persistent": 0}


def everything(b):
    b.stream.synchronize()
    keys = ("c_cell", "c_lag", "vm_cell", "c_env", "E_x", "E_y", "v_env") + (("gates",) if len(b.states[0].channel_specs) else ())
    return {k: b._dev[k].cpu().numpy().copy() for k in keys}


def far_square(b, cluster):
    """A square without membranes, in from the world's edge (which is reset every
    step): a NaN there reaches a membrane's square some steps later."""
    soff = b.offsets[2]
    ny, nx = b.worlds[cluster][1].X.shape
    sp = b._dev["sq_ptr"].cpu().numpy()
    k0 = int(soff[cluster])
    empty = [r * nx + c for r in range(2, ny - 2) for c in range(2, nx - 2)
             if sp[k0 + r * nx + c + 1] == sp[k0 + r * nx + c]]
    return k0 + empty[0]


def plant(b, cells, squares):
    for q in cells:
        b._dev["c_cell"][1, int(b.offsets[0][q]) + 3] = float("nan")
    for q in squares:
        b._dev["c_env"][0, far_square(b, q)] = float("nan")
    b.torch.cuda.synchronize()


def halted_states(worlds, flux_mode, tunings, n, cells, squares):
    runs = []
    for tuning in tunings:
        say(f"case: {len(worlds)} clusters, {flux_mode}, {n} steps, NaN in the cells of {cells}, in the env of "
            f"{squares}, tuning {tuning}")
        b = batch(worlds, flux_mode, tuning=tuning)
        b.step_n(6)
        plant(b, cells, squares)
        with pytest.raises(BetseSimUnstableException) as e:
            b.step_n(n)
        st = everything(b)
        with pytest.raises(BetseSimUnstableException) as e2:
            b.step_n(4)
        assert e2.value.step == e.value.step
        for k, v in everything(b).items():
            assert np.array_equal(v, st[k], equal_nan=True), k
        with pytest.raises(BetseSimUnstableException):
            b.step_n(5)                  # (an odd count ends with the workspace's state in the caller's buffers)
        runs.append((e.value.step, st, everything(b)))
        b.close()
    say(f"  first NaN at step {[r[0] for r in runs]}")
    for step, *states in runs[1:]:
        assert step == runs[0][0]
        for st, want in zip(states, runs[0][1:]):
            for k, v in st.items():
                assert np.array_equal(v, want[k], equal_nan=True), k
    return runs[0][0]


@pytest.mark.parametrize("n", [40, 41])
@pytest.mark.parametrize("cells,squares", [([2], []), ([], [0, 9]), ([], [5, 18])])
def test_slots_stop_at_the_first_nan(cells, squares, n):
    worlds = batched_worlds(n_clusters=19, cells_range=(10, 200), grid_range=(16, 33), seed=24)
    step = halted_states(worlds, "fp64", (SEPARATE, None), n, cells, squares)
    assert (step == 6) == bool(cells)


@pytest.mark.parametrize("n", [40, 41])
@pytest.mark.parametrize("cells,squares", [([0], []), ([], [0])])
def test_one_cluster_stops_at_its_nan(cells, squares, n):
    worlds = batched_worlds(n_clusters=1, cells_range=(60, 70), grid_range=(33, 34), seed=2)
    step = halted_states(worlds, "fp64", (SEPARATE, None, {"persistent": 1}), n, cells, squares)
    assert (step == 6) == bool(cells)


@pytest.mark.parametrize("n", [40, 41])
def test_slots_with_channels_stop_at_the_first_nan(n):
    worlds = batched_worlds(n_clusters=9, cells_range=(10, 90), grid_range=(16, 24), seed=5, base="tiny_channels")
    for p, c in worlds:
        draw_channel_state(p, c.n_cells, c.n_mems)
    assert halted_states(worlds, "fp32", (SEPARATE, None), n, [], [1, 7]) > 6


@pytest.fixture(scope="module")
def large():
    return batched_worlds(n_clusters=90, cells_range=(3800, 5000), grid_range=(100, 128), seed=11)


@pytest.mark.parametrize("n", [40, 41])
@pytest.mark.parametrize("cells,squares", [([2], []), ([80], []), ([], [3, 77])])
def test_groups_stop_at_the_first_nan(large, cells, squares, n):
    """A batch beyond the Infinity Cache, stepped in groups of clusters one after
    the other. (Separate launches skip what of the NaN's step starts after it, so the
    states to compare are those of a run without a NaN.) A step writes the workspace
    and the caller's buffers in turn, and an odd call ends in the workspace."""
    say(f"case: {len(large)} clusters in groups, {n} steps, NaN in the cells of {cells}, in the env of {squares}")
    b = batch(large, "fp64")
    b.step_n(6)
    before = everything(b)
    plant(b, cells, squares)
    with pytest.raises(BetseSimUnstableException) as e:
        b.step_n(n)
    got, off, soff = everything(b), b.offsets[0], b.offsets[2]
    b.close()
    s = e.value.step - 6
    written = s % 2 == (n + 1) % 2            # the step of the NaN wrote the buffers that the call ends in
    b = batch(large, "fp64")
    b.use_graph = False
    b.step_n(6 + s + written)
    clean = everything(b)
    b.close()
    say(f"  first NaN at step {e.value.step}")
    assert (s == 0) == bool(cells)
    for q in range(len(large)):
        if q in cells + squares:
            continue
        for k in ("c_cell", "c_lag", "vm_cell"):
            c = slice(int(off[q]), int(off[q + 1]))
            assert np.array_equal(got[k][..., c], clean[k][..., c]), (q, k)
        c = slice(int(soff[q]), int(soff[q + 1]))
        if not written:
            assert np.array_equal(got["c_env"][:, c], clean["c_env"][:, c]), q
        for k in ("v_env", "E_x", "E_y"):
            assert np.array_equal(got[k][c], before[k][c]), (q, k)


@pytest.mark.parametrize("period", [9, 10])
@pytest.mark.parametrize("n_clusters,square_of", [(1, 0), (5, 3)])
def test_sampled_loop_stops_at_the_first_nan(n_clusters, square_of, period):
    """Even and odd counts of steps before a sampled one, the NaN among them."""
    worlds = batched_worlds(n_clusters=n_clusters, cells_range=(60, 90), grid_range=(33, 36), seed=4)
    for p, _ in worlds:
        p.init_time_sampling = period * p.init_time_step
        p.set_phase_time("init")
    runs = []
    for tuning in (SEPARATE, None):
        b = batch(worlds, "fp64", tuning=tuning)
        b.step_n(6)
        plant(b, [], [square_of])
        with pytest.raises(BetseSimUnstableException) as e:
            b.run_loop(60)
        runs.append((e.value.step, everything(b)))
        b.close()
    say(f"case: {n_clusters} clusters, sampled every {period} steps, NaN at step {[r[0] for r in runs]}")
    assert runs[0][0] == runs[1][0]
    for k, v in runs[0][1].items():
        assert np.array_equal(v, runs[1][1][k], equal_nan=True), k


@pytest.mark.parametrize("n_clusters", [1, 3])
def test_a_nan_in_a_call_of_several_launches(n_clusters):
    """More steps than one launch of the persistent kernel runs."""
    worlds = batched_worlds(n_clusters=n_clusters, cells_range=(20, 60), grid_range=(12, 20), seed=4)
    assert halted_states(worlds, "fp64", (SEPARATE, None), 9001, [], [n_clusters - 1]) < 40
