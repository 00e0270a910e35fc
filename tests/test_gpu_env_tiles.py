"""The environment kernel where its tiles, staged pairs and stencils end: grids
around multiples of the 16x16 tile (the last tile one to three squares wide, odd
and even widths, grids whose tiles all touch the world's edge and grids with
inner ones), a D_env that is one value and one that varies over the squares,
with the exchange in the kernel and in a launch of its own, and the fluxes of an
observed step. Bars: those of the FP64 parity tests; a flux's two terms are a
difference of two concentrations (each within the concentrations' bar) over the
grid spacing and the field (within E's bar) times one."""

import numpy as np
import pytest

from betse_amd.cells import Cells
from betse_amd.parameters import Parameters
from tests.test_gpu_parity import E_TOL, REL_TOL, check, oracle_run, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("varying", [False, True], ids=["uniform", "varying"])
@pytest.mark.parametrize("grid", [16, 17, 18, 19, 31, 33, 34, 35, 49, 52])
def test_env_tiles(grid, varying):
    from betse_amd.sim import SimPhase, SimPhaseKind, Simulator
    p = Parameters.preset("tiny")
    p.grid_size = grid
    if varying:
        p.D_adh, p.D_tj = 0.5, 0.1
    cells = Cells.make_world(p)
    say(f"case: {grid}x{grid} grid, D_env {'varying' if varying else 'uniform'}")
    n = 21
    before = oracle_run(p, cells, n)
    after = oracle_run(p, cells, n + 1)
    for tuning in ({"exchange_form": 2, "env_ions_per_block": 5}, {"exchange_form": 0, "env_ions_per_block": 2}):
        sim = Simulator(p.copy(), device="cuda:0", flux_mode="fp64", tuning=tuning)
        phase = SimPhase(SimPhaseKind.INIT, sim.p, cells, sim)
        sim.init_core(phase)
        sim.prepare(phase)
        sim.step_n(n)
        sim.pull()
        check(sim, before, f"  {tuning}")
        sim.step_observed(1)
        sim.pull_raw_fluxes()
        check(sim, after, "  observed step")
        for name in ("fluxes_env_x", "fluxes_env_y"):
            ref, got = np.asarray(getattr(after, name)), getattr(sim, name)
            D = np.asarray(after.D_env).max(axis=1)
            bar = D * np.asarray(after.cc_env).max(axis=1) * 2.0 * REL_TOL / cells.delta
            bar = bar + E_TOL * np.abs(ref).max(axis=1)
            assert (np.abs(got - ref).max(axis=1) <= bar).all(), name
