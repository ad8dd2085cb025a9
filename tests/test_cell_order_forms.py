"""The forms of positions that the cell order takes and refuses: wider rows give
the order of their first three columns, grids beyond 2048 cells theirs."""
import numpy as np
import pytest

from diffskill_amd.engine.core import cell_order, cell_sort_perm


def _order(x, n_grid):
    b = np.clip(np.trunc(x[:, :3] * n_grid - 0.5).astype(np.int64), 0, n_grid - 1)
    nb = (n_grid + 3) // 4
    blk = ((b[:, 0] >> 2) * nb + (b[:, 1] >> 2)) * nb + (b[:, 2] >> 2)
    cell = ((b[:, 0] & 3) << 4) | ((b[:, 1] & 3) << 2) | (b[:, 2] & 3)
    return np.argsort(blk * 64 + cell, kind="stable")


@pytest.mark.parametrize("width", [3, 4, 6, 9])
@pytest.mark.parametrize("n", [0, 1, 2, 500])
def test_wide_rows(n, width):
    x = np.random.default_rng(n + width).random((n, width))
    for form in (x, np.asfortranarray(x), x[::-1][::-1]):
        assert np.array_equal(cell_sort_perm(form, 64), _order(x, 64))
    if n:
        assert np.array_equal(cell_sort_perm(x.astype(np.float32), 64), _order(x.astype(np.float32).astype(np.float64), 64))


@pytest.mark.parametrize("n_grid", [2048, 2049, 5000, 70000])
def test_fine_grids(n_grid):
    x = np.random.default_rng(n_grid).uniform(-0.1, 1.1, (800, 3))
    x[100:200] = x[:100]
    perm, inv = cell_order(x, n_grid)
    assert np.array_equal(perm, _order(x, n_grid)) and np.array_equal(inv[perm], np.arange(800))


def test_refused():
    for bad in (np.zeros(3), np.zeros((4, 2)), np.zeros((2, 3, 3))):
        with pytest.raises((ValueError, IndexError)):
            cell_sort_perm(bad, 64)
    x = np.zeros((5, 6))
    for out in (np.empty((2, 4), np.int64), np.empty((2, 5), np.int32), np.empty((5, 2), np.int64).T):
        with pytest.raises(ValueError):
            cell_order(x, 64, out)
