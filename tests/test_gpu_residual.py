"""The per-cluster residual of a window against numpy on the states before and after:
clusters smaller than a wavefront, clusters that end inside one, a last wavefront that
is not full, and a NaN (infinite residual of its cluster only)."""

import ctypes

import numpy as np
import pytest

from betse_amd.batch import batched_worlds
from tests.test_gpu_configs import batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells", [(1, (3, 6)), (9, (3, 130)), (5, (200, 700))])
def test_residual_matches_numpy(n, cells):
    b = batch(batched_worlds(n_clusters=n, cells_range=cells, grid_range=(8, 48), seed=n), "fp64")
    off = b.offsets[0]
    print(f"{n} clusters, {off[-1]} cells", flush=True)
    c0, _ = b.snapshot()
    r = b.residual_window(3)
    c1, _ = b.snapshot()
    d = np.abs(c1 - c0)
    rel = np.where(c1 != 0.0, d / np.where(c1 != 0.0, np.abs(c1), 1.0), d).max(axis=0)
    want = np.array([rel[off[i]:off[i + 1]].max() for i in range(n)])
    assert np.array_equal(r, want / 3.0)
    torch = b.torch
    prev = torch.tensor(c0, device=b.device)
    prev[0, int(off[n - 1])] = float("nan")
    out = torch.empty(n, dtype=torch.float64, device=b.device)
    torch.cuda.synchronize()
    assert b._lib.bt_residual(b._ctx, ctypes.c_void_p(prev.data_ptr()),
                              ctypes.c_void_p(b._dev["cell_cluster"].data_ptr()),
                              ctypes.c_void_p(out.data_ptr())) == 0
    b.sync()
    out = out.cpu().numpy()
    assert out[n - 1] == np.inf and np.array_equal(out[:n - 1], want[:n - 1])
    b.close()
