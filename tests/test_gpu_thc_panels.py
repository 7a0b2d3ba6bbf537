"""Edges of the grid pruning's steps: blocks around the 128 vectors that a
panel of the Schur form holds, candidate counts around the 64 of a workgroup,
and the on-the-fly form, against the oracle's pivot sequence (exact)."""
import numpy as np
import pytest

import thc as thc_oracle
from gigpu import lib, systems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case():
    b = systems.water_system(1, 6.0, "small", seed=3)
    c = lib.Context(0)
    c.set_basis(b)
    pts = systems.atom_centred_points(b, radii=(0.2, 0.5, 0.9, 1.5, 2.4, 3.6), ndir=30, seed=8)   # 540 points
    yield c, b, pts
    c.close()


@pytest.mark.parametrize("block", [1, 60, 127, 128, 129, 200, 256, 257, 500])
def test_block_sizes(case, block):
    c, b, pts = case
    ref, nred = thc_oracle.grid_pivots(b, pts, 1e-4, 1e-3, block)
    got, gred = c.thc_grid_pivots(pts, 1e-4, 1e-3, block)
    assert len(ref) > 128 or block < 128
    assert gred == nred and np.array_equal(got, ref)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 321])
@pytest.mark.parametrize("schur_mb", [24576, 0])
def test_candidate_counts(case, n, schur_mb):
    c, b, pts = case
    ref, nred = thc_oracle.grid_pivots(b, pts[:n], 1e-3, -1.0, 100)
    c.set_option("thc_schur_mb", schur_mb)
    try:
        got, gred = c.thc_grid_pivots(pts[:n], 1e-3, -1.0, 100)
    finally:
        c.set_option("thc_schur_mb", 24576)
    assert gred == nred and np.array_equal(got, ref)


@pytest.mark.parametrize("n", [1023, 1025, 2160])
def test_block_columns(case, n):
    """Candidates around the 1024 columns of a block column of the Schur form."""
    c, b, _ = case
    pts = systems.atom_centred_points(b, radii=(0.2, 0.5, 0.9, 1.5, 2.4, 3.6), ndir=120, seed=8)[:n]
    ref, nred = thc_oracle.grid_pivots(b, pts, 1e-3, 1e-2, 200)
    got, gred = c.thc_grid_pivots(pts, 1e-3, 1e-2, 200)
    assert gred == nred and np.array_equal(got, ref)
