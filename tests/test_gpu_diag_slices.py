"""Diagonals of contracted pairs, whose slices of sixteen columns are tiles of
their own, against the oracle's (pq|pq): 1 to 7 slices ((ff) has 28 and 49
spherical, 55 and 100 Cartesian columns), in classes that mix pairs with and
without contractions and, with a second molecule, pairs of fewer columns."""
import numpy as np
import pytest

from gigpu import systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,spher", [(1, True), (1, False), (2, True)])
def test_vdiag(gpu_ctx, oracle_mod, waters, spher):
    b = systems.water_system(waters, 6.0, "large", seed=17, contracted=True, spher_ao=spher)
    gpu_ctx.set_basis(b)
    gpu_ctx.chol_build(tau=1e-2, flags=1)
    ref = oracle_mod.Oracle(b).chol(tau=1e-2, flags=1)
    assert ref.status == 0, ref.message
    assert np.abs(gpu_ctx.chol_vdiag() - ref.vdiag).max() <= 1e-12
