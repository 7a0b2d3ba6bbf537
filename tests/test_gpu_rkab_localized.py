"""Rkab of orbitals and vectors that decay over space, at sizes of large
products: every element is exact to the rounding of its own terms, the tiny
ones of distant supports too.  The bar is that of an FP64 sum in any order,
(k + 1) 2^-53 sum |Z| |Xa Xb|."""
import numpy as np
import pytest

from gigpu import lib, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("decay", [0.1, 0.3])
def test_elements_of_distant_supports(decay):
    b = systems.water_system(8, 7.9, "large", seed=2)   # 600 AOs, for their number
    n, nv, na, nb = 1700, 3400, 40, 500
    rng = np.random.default_rng(11)
    pg, po, pk = 20.0 * rng.random(n), 20.0 * rng.random(b.nao), 20.0 * rng.random(nv)   # on a line of 20 bohr
    X = np.asfortranarray(np.exp(-decay * (pg[:, None] - po) ** 2) * rng.standard_normal((n, b.nao)))
    Z = np.asfortranarray(np.exp(-decay * (pg[:, None] - pk) ** 2) * rng.standard_normal((n, nv)))
    C = np.asfortranarray(np.eye(b.nao))   # orbitals are columns of X, to the last bit
    c = lib.Context(0)
    try:
        c.set_basis(b)
        got = c.thc_rkab(X, Z, C, 1, na, C, na + 1, na + nb, 0).reshape(nv, na, nb, order="F")
    finally:
        c.close()
    k, a, q = rng.choice(nv, 40, replace=False), rng.integers(0, na, 60), rng.integers(0, nb, 60)
    A, B = Z[:, k].T, (X[:, a] * X[:, na + q]).T
    ref = np.asarray(A, np.longdouble) @ np.asarray(B, np.longdouble).T
    err = np.abs(got[np.ix_(k, range(na), range(nb))][:, a, q] - ref).astype(float)
    bar = (n + 1) * 2.0 ** -53 * (np.abs(A) @ np.abs(B).T)
    assert (err <= bar).all(), float((err / bar).max())
