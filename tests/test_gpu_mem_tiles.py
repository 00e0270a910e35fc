"""The membrane kernel where its tiles' (ion, cell) items end: cells of 3 to 10
membranes (tiles of few and of many cells, one pass of a wavefront over the items
and several), three to seven ions, one and two wavefronts per tile. Bars: those of
the FP64 parity tests."""

import numpy as np
import pytest

from betse_amd.cells import Cells
from betse_amd.parameters import Parameters
from tests.test_gpu_parity import check, oracle_run, say

pytestmark = pytest.mark.gpu

CELL = {"Na": 8.0, "K": 125.0, "Cl": 10.0, "Ca": 1.0e-4, "H": 6.0e-5, "P": 100.0}
ENV = {"Na": 145.0, "K": 5.0, "Cl": 105.0, "Ca": 1.0, "H": 4.0e-5, "P": 10.0}


@pytest.mark.parametrize("ions", [("Na", "K"), ("Na", "K", "P"), ("Na", "K", "Cl", "Ca", "P"),
                                  ("Na", "K", "Cl", "Ca", "H", "P")], ids=lambda i: f"{len(i) + 1}ions")
def test_mem_tiles(ions):
    p = Parameters.preset("tiny")
    p.set_ion_profile({n: CELL[n] for n in ions}, {n: ENV[n] for n in ions},
                      {"Na": 1.0e-18, "K": 15.0e-18, "Cl": 2.0e-18})
    p.init_time_step = 1.0e-4
    p.set_phase_time("init")
    rng = np.random.RandomState(5)
    cells = Cells.make_world(p, points=rng.uniform(-60e-6, 60e-6, (500, 2)))
    say(f"case: ions {ions}, cells of {cells.num_mems.min()}-{cells.num_mems.max()} membranes")
    n = 11
    o = oracle_run(p, cells, n)
    from betse_amd.sim import SimPhase, SimPhaseKind, Simulator
    for waves in (1, 2):
        sim = Simulator(p.copy(), device="cuda:0", flux_mode="fp64", tuning={"mem_waves": waves})
        phase = SimPhase(SimPhaseKind.INIT, sim.p, cells, sim)
        sim.init_core(phase)
        sim.prepare(phase)
        sim.step_n(n)
        sim.pull()
        check(sim, o, f"  mem_waves {waves}")
