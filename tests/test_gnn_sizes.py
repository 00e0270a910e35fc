"""The network's size functions take any count: they run on the host, without a GPU."""

import os

import pytest

from betse_amd import _native


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built (run __graft_entry__.build())")
    return _native.load()


@pytest.mark.parametrize("n", [0, -1, -4097])
def test_no_nodes_need_no_workspace(lib, n):
    assert lib.bt_gnn_backward_len(16, 4, 32, 3, n) == 0


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 4097, 262_145, 1 << 24])
def test_workspace_holds_what_a_pass_keeps(lib, n):
    f_in, f_out, H, L = 16, 4, 32, 3
    splits = min(64, -(-n // 4096)) if n > 4096 else 1
    chunk = -(-(-(-n // splits)) // 16) * 16
    splits = -(-n // chunk)
    weights = f_in * H + 2 * L * H * H + H * f_out
    assert lib.bt_gnn_backward_len(f_in, f_out, H, L, n) == (
        n * H * (L + 4) + splits * weights + -(-n // 256) * (H * (L + 1) + f_out))
