"""The exchange of squares whose membranes take one, two and three loads of four (and
none), with and without a channel's row: bit for bit the per-square form's result."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
@pytest.mark.parametrize("base", ["tiny", "tiny_channels"])
def test_exchange_rows(base, flux_mode):
    worlds = batched_worlds(n_clusters=3, cells_range=(40, 300), grid_range=(6, 16), seed=8, base=base)
    if base == "tiny_channels":
        from betse_amd.channels import draw_channel_state
        for p, c in worlds:
            draw_channel_state(p, c.n_cells, c.n_mems)
    per_square = np.concatenate([np.bincount(c.map_mem2ecm, minlength=c.X.size) for _, c in worlds])
    assert {min(3, -(-int(m) // 4)) for m in per_square} == {0, 1, 2, 3}
    runs = []
    for form in (0, 1):
        say(f"case: {base}, {flux_mode}, exchange form {form}, up to {per_square.max()} membranes per square")
        b = batch(worlds, flux_mode, tuning={"exchange_form": form, "persistent": 0})
        b.step_n(11)
        runs.append(state(b))
        b.close()
    for k in runs[0]:
        assert np.array_equal(runs[0][k], runs[1][k]), k
