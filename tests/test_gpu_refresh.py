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


@pytest.mark.parametrize("tuning", [{"persistent": 0}, None], ids=["graphs", "default"])
def test_refresh_takes_the_geometry_again(monkeypatch, tuning):
    """Volumes and gap-junction partners changed in the caller's buffers: the steps
    are those of a context created with them."""
    import betse_amd.batch as module
    worlds = batched_worlds(n_clusters=2, cells_range=(30, 60), grid_range=(16, 20), seed=5)
    say(f"case: cell_vol and nn_mem changed, tuning {tuning}")

    def changed(geo):
        m = int(np.flatnonzero(geo["nn_mem"] != np.arange(len(geo["nn_mem"])))[0])
        geo["nn_mem"][m] = m                    # one membrane's gap junction closed for good
        geo["nn_cell"][m] = geo["mem_cell"][m]
        geo["cell_vol"] *= 1.25
        return geo

    b = batch(worlds, "fp64", tuning=tuning)
    for k, v in changed({k: b._dev[k].cpu().numpy().copy() for k in ("nn_mem", "nn_cell", "mem_cell", "cell_vol")}).items():
        b._dev[k].copy_(b.torch.from_numpy(v))
    b.torch.cuda.synchronize()
    b.set_membrane_params(0)
    b.step_n(21)
    got = state(b)
    b.close()
    plain = module.batch_geometry
    monkeypatch.setattr(module, "batch_geometry", lambda cells: (lambda g, o: (changed(g), o))(*plain(cells)))
    b = batch(worlds, "fp64", tuning=tuning)
    b.step_n(21)
    want = state(b)
    b.close()
    for k in want:
        assert np.array_equal(got[k], want[k]), k
