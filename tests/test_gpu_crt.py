"""Large products on the int8 matrix cores (crt.hip), where a decomposition or
a THC fit takes them: the vectors Inv_L V(P, pq) of (H2O)6 and the THC fit's
right-hand side, against the same products in extended precision.

The bar is the scheme's own: a scaled row has a norm of 2^57..2^58 units and
each element is off by half a unit, so an element of A B^T with k terms is off
by at most sqrt(k) 2^-57 |a| |b|, plus one rounding of the result."""
import numpy as np
import pytest

from gigpu import lib, systems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def built():
    b = systems.water_system(6, 7.2, "large", seed=41)
    c = lib.Context(0)
    c.set_basis(b)
    c.chol_build(tau=1e-5)
    yield c, b, c.chol_meta(), c.chol_rkpq()
    c.close()


def _exact(A, B):
    """A B^T in extended precision (64-bit mantissa)."""
    return np.asarray(A, np.longdouble) @ np.asarray(B, np.longdouble).T


def _bar(A, B, ref):
    k = A.shape[1]
    return (np.sqrt(k) * 2.0 ** -57 * np.linalg.norm(A, axis=1)[:, None] * np.linalg.norm(B, axis=1)[None, :]
            + 2.0 ** -52 * np.abs(ref) + np.sqrt(k) * 2.0 ** -63 * (np.abs(A) @ np.abs(B).T)).astype(float)


def test_vectors(built):
    c, b, m, R = built
    X = c.chol_inv_l()
    nv = m["nvecs"]
    assert nv > 2000 and nv % 256 != 0   # the route and ragged tiles
    sp, loc = m["shell_pairs"], m["shell_pair_loc"]
    piv = [tuple(sp[i - 1] - 1) for i in m["pivot_shell_pairs"]]
    sel, off, k = [], 0, 0
    for (p, q), n in zip(piv, m["pivot_shell_pair_dim"]):
        sel += [off + m["pivot_orb_pairs"][k + j] - 1 for j in range(n)]
        k += n
        off += b.shell_nang(p) * b.shell_nang(q)
    rng = np.random.default_rng(1)
    ends = [0, 1, len(sp) - 2, len(sp) - 1]
    pick = [s for s in ends + list(rng.choice(len(sp), 12, replace=False)) if sp[s][0] != sp[s][1]]
    V = c.eri_pair_block([tuple(sp[s] - 1) for s in pick], piv)[:, sel]
    got = np.concatenate([R[loc[s][2] - 1, loc[s][1] - 1:loc[s][1] - 1 + m["shell_pair_dim"][s]] for s in pick])
    rows = np.unique(np.concatenate([[0, 1, 255, 256, 257, nv - 2, nv - 1], rng.choice(nv, 60, replace=False)]))
    ref = _exact(X[rows], V)
    err = np.abs(got.T[rows] - ref)
    assert (err <= _bar(X[rows], V, ref)).all(), float((err / _bar(X[rows], V, ref)).max())


def test_thc_right_hand_side(built):
    """Z of a well-conditioned grid: S Z = XR recovers XR, whose rows are the
    folded products over the stored columns."""
    c, b, m, R = built
    pts = systems.atom_centred_points(b, radii=(0.4, 1.0, 2.4), ndir=24, seed=3)   # 1296 points: the int8 route
    X = c.thc_orbitals(pts)
    Z, _ = c.thc_z(X)
    S = (X @ X.T) ** 2
    XR = S @ Z
    loc0 = np.concatenate([[0], np.cumsum([b.shell_nang(s) for s in range(b.nshells)])])
    g = np.array([0, 1, 255, 256, 300, len(pts) - 1])
    ref = np.zeros((len(g), m["nvecs"]))
    for (A, B), (_, pos, sub) in zip(m["shell_pairs"], m["shell_pair_loc"]):
        na, nb = b.shell_nang(A - 1), b.shell_nang(B - 1)
        ab = [(i, j) for j in range(nb) for i in range(j if A == B else 0, na)]
        P = np.array([loc0[A - 1] + i for i, _ in ab])
        Q = np.array([loc0[B - 1] + j for _, j in ab])
        w = np.where(P == Q, 1.0, 2.0)
        ref += (X[np.ix_(g, P)] * X[np.ix_(g, Q)] * w) @ R[sub - 1, pos - 1:pos - 1 + len(ab)]
    # Z = L^-T (L^-1 XR) leaves a residual of eps cond(L) |S| |Z|, cond(L) below 1e4 on such grids
    bar = 1e-11 * (np.abs(S[g]) @ np.abs(Z)).max()
    assert np.abs(XR[g] - ref).max() <= bar


def test_non_finite_points_are_not_scaled(built):
    """A point with an infinite orbital value cannot be scaled to integers: the
    call takes the DGEMM route and ends as it did there (an error for the
    metric, or non-finite numbers), and the context stays usable."""
    c, b, m, R = built
    pts = systems.atom_centred_points(b, radii=(0.4, 1.0, 2.4), ndir=24, seed=3)
    X = c.thc_orbitals(pts)
    Y = X.copy(order="F")
    Y[7, 3] = np.inf
    try:
        Z, _ = c.thc_z(Y)
        assert not np.isfinite(Z).all()
    except lib.GigpuError:
        pass
    Z, _ = c.thc_z(X)
    assert np.isfinite(Z).all()


@pytest.mark.parametrize("points,nvec,na,nb", [(2177, 2817, 40, 300), (900, 6001, 100, 200), (1999, 4099, 25, 425)])
def test_rkab_products(built, points, nvec, na, nb):
    """Rkab = Z^T (Xa o Xb) at ragged tiles, sampled against extended precision."""
    c, b, _, _ = built
    rng = np.random.default_rng(points)
    X = np.asfortranarray(rng.standard_normal((points, b.nao)) * np.exp(-20.0 * rng.random((points, b.nao)) ** 2))
    Z = np.asfortranarray(rng.standard_normal((points, nvec)))
    C = np.asfortranarray(np.eye(b.nao)[:, rng.permutation(b.nao)])   # orbitals are columns of X, to the last bit
    got = c.thc_rkab(X, Z, C, 1, na, C, na + 1, na + nb, 0).reshape(nvec, na, nb, order="F")
    Y = X @ C
    k = np.unique(np.concatenate([[0, 255, 256, nvec - 1], rng.choice(nvec, 30, replace=False)]))
    a, q = rng.integers(0, na, 40), rng.integers(0, nb, 40)
    a[:2], q[:2] = [0, na - 1], [0, nb - 1]
    A, B = Z[:, k].T, (Y[:, a] * Y[:, na + q]).T
    ref = _exact(A, B)
    assert (np.abs(got[np.ix_(k, range(na), range(nb))][:, a, q] - ref) <= _bar(A, B, ref)).all()
