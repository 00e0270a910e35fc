"""The persistent kernel's forms against replayed graphs and separate launches, bit
for bit: one wavefront per cell tile (more tiles than its blocks take with three),
the ordered phases of a Ca pump and of channels, by size or forced."""

import numpy as np
import pytest

from betse_amd.batch import BatchSimulator, batched_worlds
from betse_amd.cells import Cells
from betse_amd.channels import draw_channel_state
from betse_amd.parameters import Parameters
from tests.test_gpu_configs import say, state

pytestmark = pytest.mark.gpu

GRAPHS, TEAM = {"persistent": 0}, {"persistent": 1}


def compare_forms(worlds, flux_mode, forms, counts=(1, 2, 21)):
    runs = []
    for tuning, use_graph, persistent in forms:
        b = BatchSimulator([(p.copy(), c) for p, c in worlds], device="cuda:0", flux_mode=flux_mode, tuning=tuning,
                           use_graph=use_graph)
        b.init("init")
        say(f"case: {b.n_cells} cells in {b.n_tiles} tiles, {flux_mode}, tuning {tuning}, graphs {use_graph}")
        assert b.running_tuning()["persistent"] == persistent
        for n in counts:
            b.step_n(n)
        st = state(b)
        keys = ("v_env",) + (("gates",) if len(b.states[0].channel_specs) else ())
        st.update({k: b._dev[k].cpu().numpy() for k in keys})
        runs.append((b.n_tiles, st))
        b.close()
    for _, r in runs[1:]:
        for k in runs[0][1]:
            assert np.array_equal(runs[0][1][k], r[k]), k
    return runs[0][0]


ALL = [(None, True, 1), (GRAPHS, True, 0), (None, False, 0), (TEAM, False, 1)]


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
@pytest.mark.parametrize("cells,grid", [((1420, 1460), (50, 51)),          # 16 env tiles: 16 blocks for the cells
                                        ((1240, 1300), (44, 45))])         # 9 env tiles: 23
def test_one_wavefront_per_tile(cells, grid, flux_mode):
    worlds = batched_worlds(n_clusters=1, cells_range=cells, grid_range=grid, seed=31)
    assert compare_forms(worlds, flux_mode, ALL) > 5 * (16 if grid[0] > 48 else 23)


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
@pytest.mark.parametrize("n_clusters", [1, 11])
def test_calcium_pump(n_clusters, flux_mode):
    worlds = batched_worlds(n_clusters=n_clusters, cells_range=(30, 150), grid_range=(16, 34), seed=6)
    for p, _ in worlds:
        p.set_ion_profile({"Na": 8.0, "K": 125.0, "Cl": 10.0, "Ca": 1e-4, "P": 100.0},
                          {"Na": 145.0, "K": 5.0, "Cl": 105.0, "Ca": 1.0, "P": 10.0},
                          {"Na": 1e-18, "K": 15e-18, "Cl": 2e-18})
    compare_forms(worlds, flux_mode, ALL)


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
@pytest.mark.parametrize("n_clusters,cells,grid", [(3, (30, 200), (16, 24)), (1, (1700, 1800), (33, 34))])
def test_channels(n_clusters, cells, grid, flux_mode):
    """With more tiles than the blocks take with three wavefronts each only where
    the persistent kernel is forced."""
    worlds = batched_worlds(n_clusters=n_clusters, cells_range=cells, grid_range=grid, seed=5, base="tiny_channels")
    for p, c in worlds:
        draw_channel_state(p, c.n_cells, c.n_mems)
    small = n_clusters > 1
    tiles = compare_forms(worlds, flux_mode, ALL if small else [(TEAM, True, 1), (GRAPHS, True, 0), (None, False, 0)])
    assert small or tiles > 160


@pytest.mark.parametrize("flux_mode", ["fp64", "fp32"])
def test_channels_of_triangular_cells(flux_mode):
    """Tiles of 21 cells (three membranes each) with three channels: a block's LDS
    holds fewer tiles than it has wavefronts."""
    p = Parameters.preset("tiny_full")
    p.network, p.cluster_radius, p.grid_size = None, 380e-6, 33
    a, n = 10e-6, 44                      # cells around the vertices of a honeycomb
    i, j = np.meshgrid(np.arange(-n, n), np.arange(-n, n), indexing="ij")
    x, y = 1.5 * a * i.ravel(), np.sqrt(3) * a * (j + 0.5 * (i % 2)).ravel()
    cells = Cells.make_world(p, points=np.stack([np.concatenate([x, x + a]), np.concatenate([y, y])], axis=1))
    assert set(cells.num_mems.tolist()) == {3}
    draw_channel_state(p, cells.n_cells, cells.n_mems)
    assert compare_forms([(p, cells)], flux_mode, [(TEAM, True, 1), (GRAPHS, True, 0), (None, False, 0)]) > 160
