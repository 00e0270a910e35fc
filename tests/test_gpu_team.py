"""Small problems step in one kernel per call, a team of blocks per XCD sharing
out the clusters. Its states, fields and halt are those of the replayed
three-kernel steps bit for bit, over step counts of either parity, clusters of a
single tile, more clusters than XCDs, and the ordered phases of the Ca pump."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from betse_amd.exceptions import BetseSimUnstableException
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu

GRAPHS = {"persistent": 0}          # setting any tuning leaves the default choice
CASES = [dict(n_clusters=1, cells_range=(3, 6), grid_range=(8, 10)),        # one tile, one block of work
         dict(n_clusters=1, cells_range=(60, 70), grid_range=(33, 34)),     # env tiles of one row
         dict(n_clusters=7, cells_range=(4, 90), grid_range=(8, 40)),
         dict(n_clusters=19, cells_range=(10, 200), grid_range=(16, 33)),   # several clusters to a slot
         dict(n_clusters=3, cells_range=(500, 900), grid_range=(16, 48))]   # more tiles than wavefronts


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_team_steps_are_bit_identical(case, flux_mode):
    worlds = batched_worlds(seed=21 + case, **CASES[case])
    runs = []
    for tuning in (None, GRAPHS, {"persistent": 1}):
        say(f"case: {CASES[case]}, {flux_mode}, tuning {tuning}")
        b = batch(worlds, flux_mode, tuning=tuning)
        for n in (1, 2, 3, 36):
            b.step_n(n)
        st = state(b)
        st.update({k: b._dev[k].cpu().numpy() for k in ("v_env", "E_x", "E_y")})
        runs.append(st)
        b.close()
    for r in runs[1:]:
        for k in runs[0]:
            assert np.array_equal(runs[0][k], r[k]), k


@pytest.mark.parametrize("n", [20, 21])
@pytest.mark.parametrize("tuning", [None, GRAPHS], ids=["team", "graphs"])
def test_team_halts_at_the_step_of_the_nan(tuning, n):
    worlds = batched_worlds(n_clusters=11, cells_range=(30, 200), grid_range=(16, 40), seed=3)
    say(f"case: NaN in cluster 9, {n} steps, tuning {tuning}")
    b = batch(worlds, "fp64", tuning=tuning)
    b.step_n(6)
    b._dev["c_cell"][1, int(b.offsets[0][9]) + 3] = float("nan")
    for _ in range(2):
        with pytest.raises(BetseSimUnstableException) as e:
            b.step_n(n)
        assert e.value.step == 6
    b.close()
