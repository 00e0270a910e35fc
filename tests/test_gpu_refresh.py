"""A refused change of the membranes' or the environment's values leaves the
context as it was: the steps after it, and after the change is made acceptable,
are those of a context that never saw the refusal, bit for bit."""

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from betse_amd.channels import draw_channel_state
from betse_amd.exceptions import BetseNativeError
from tests.test_gpu_configs import batch, say, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tuning", [{"persistent": 0}, None], ids=["graphs", "default"])
def test_steps_after_a_refused_change(tuning):
    worlds = batched_worlds(n_clusters=2, cells_range=(30, 60), grid_range=(16, 20), seed=5, base="tiny_channels")
    for p, c in worlds:
        draw_channel_state(p, c.n_cells, c.n_mems)
    say(f"case: D_env that varies with a refused Phi_b, tuning {tuning}")
    runs = []
    for refused in (False, True):
        b = batch(worlds, "fp64", tuning=tuning)
        b.step_n(4)
        s0, s1 = int(b.offsets[2][1]), int(b.offsets[2][2])
        D = b._dev["D_env"][:, s0:s1].cpu().numpy().copy()
        D[:, ::3] *= 0.5
        if refused:
            b._dev["Phi_b"][s0] = 0.01
            b.torch.cuda.synchronize()
            with pytest.raises(BetseNativeError, match="Phi_b"):
                b.set_membrane_params(1, D_env=D)
            b._dev["Phi_b"].zero_()
            b.torch.cuda.synchronize()
        b.set_membrane_params(1, D_env=D)
        b.step_n(21)
        runs.append(state(b))
        b.close()
    for k in runs[0]:
        assert np.array_equal(runs[0][k], runs[1][k]), k
