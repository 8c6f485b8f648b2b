"""Products with few vectors at the sizes where their loops and copies change, against the
reference's sum (ascending beamlets, float64, product rounded before the add) bit for bit."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dij(n_rows, per_row, n_cols, seed=0):
    """Rows in turn with per_row[i % len] entries of random columns."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for r in range(n_rows):
        k = per_row[r % len(per_row)]
        rows += [r] * k
        cols += sorted(rng.choice(n_cols, size=k, replace=False).tolist())
    order = np.lexsort((rows, cols))
    rows, cols = np.array(rows, np.int64)[order], np.array(cols, np.int64)[order]
    indptr = np.concatenate(([0], np.cumsum(np.bincount(cols, minlength=n_cols)))).astype(np.int64)
    return SimpleNamespace(indptr=indptr, indices=rows, dose=rng.standard_normal(rows.size), n_beamlets=n_cols,
                           n_voxels=n_rows, grid_shape=(n_rows, 1, 1)), cols


# Blocks with no entry, around the number of entries loaded ahead (4 to 16) and beyond it; a
# row count off the block; products below and above the staged size (1 MiB).
@pytest.mark.parametrize("n_w", (1, 2, 3, 4, 5, 8))
@pytest.mark.parametrize("n_rows, per_row", [(13, (0,)), (21, (3, 0, 1, 16, 0, 2, 17, 4)), (75, (15, 33)),
                                             (140_000, (1, 0, 2))])
def test_few_vectors_match_the_reference_sum(n_w, n_rows, per_row):
    from pyradmc_amd.spmm import DeviceDij

    dij, cols = _dij(n_rows, per_row, 40)
    weights = np.random.default_rng(1).standard_normal((40, n_w))
    weights[3, 0] = np.inf  # only rows that hold the beamlet see it
    want = np.zeros((n_rows, n_w))
    np.add.at(want, dij.indices, dij.dose[:, None] * weights[cols])
    dev = DeviceDij(dij)
    np.testing.assert_array_equal(dev.apply(weights), want)
    np.testing.assert_array_equal(dev.apply(weights, rows=(5, n_rows - 1)), want[5:-1])
    got = dev.apply_transpose(np.arange(n_rows, dtype=np.float64))
    ref = np.zeros(40)
    np.add.at(ref, cols, dij.dose * dij.indices)
    np.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-11 * max(np.abs(ref).max(), 1.0))
    dev.close()


def test_refused_products_allocate_nothing():
    """Row ranges outside the matrix and products beyond one launch are refused as such,
    whatever memory their result would have taken."""
    from pyradmc_amd.spmm import DeviceDij

    dij, _ = _dij(21, (3, 0, 1), 40)
    dev = DeviceDij(dij)
    weights = np.ones(40)
    for rows in ((0, 10**13), (-(10**13), 5), (5, 5), (6, 5), (0, 22)):
        for fetch in (True, False):
            with pytest.raises(ValueError, match="row range"):
                dev.apply(weights, rows=rows, fetch=fetch)
    with pytest.raises(ValueError):
        dev.apply(np.ones((40, 0)))
    assert dev.apply(weights).shape == (21,)
    dev.close()
