"""Edges of the first MO step's tiles (k_mo_half): numbers of MO columns at
and around the multiples of four and of the widest wave (80), several waves,
vector counts below and not a multiple of 64, pair lists shorter than a chunk,
and passes of a few columns, against a dense product of the same vectors.  A
component is a sum of at most nao^2 products of factors exact to rounding:
1e-12 of the largest component."""
import numpy as np
import pytest

from gigpu import lib, systems
from gigpu.basis import build_basis

pytestmark = pytest.mark.gpu


def _dense(ctx, basis):
    """L^k (nvec, nao, nao) from the library's vectors."""
    m, R = ctx.chol_meta(), ctx.chol_rkpq()
    loc = np.concatenate([[0], np.cumsum([basis.shell_nang(s) for s in range(basis.nshells)])])
    L = np.zeros((m["nvecs"], basis.nao, basis.nao))
    for (A, B), (_, pos, X) in zip(m["shell_pairs"], m["shell_pair_loc"]):
        na, nb, q = basis.shell_nang(A - 1), basis.shell_nang(B - 1), 0
        for b in range(nb):
            for a in range(b if A == B else 0, na):
                p, r = loc[A - 1] + a, loc[B - 1] + b
                L[:, p, r] = L[:, r, p] = R[X - 1, pos - 1 + q]
                q += 1
    return L


def _tiny():
    shells = {"H": [(0, [0.3], [1.0]), (0, [1.7], [1.0]), (1, [0.8], [1.0])]}
    return build_basis(["H", "H"], np.array([[0.0, 0.0, 0.0], [0.9, 0.3, -0.2]]), shells)


@pytest.fixture(scope="module", params=["tiny", "water", "waters"])
def case(request):
    b = {"tiny": _tiny, "water": lambda: systems.water_system(1, 6.0, "small", seed=9),
         "waters": lambda: systems.water_system(2, 6.0, "small", seed=9)}[request.param]()
    c = lib.Context(0)
    c.set_basis(b)
    c.chol_build(tau=1e-6)
    yield c, b, _dense(c, b)
    c.close()


@pytest.mark.parametrize("na", [1, 3, 4, 5, 12, 13, 31, 37, 40, 41, 79, 80, 81, 96, 161])
def test_column_counts(case, na):
    ctx, b, L = case
    rng = np.random.default_rng(na)
    C, D = rng.normal(size=(b.nao, na)), rng.normal(size=(b.nao, 3))
    ref = np.matmul(np.matmul(C.T, L), D)   # (k, a, b)
    got = ctx.mo_transform(C, 1, na, D, 1, 3, flags=lib.MO_ALL_COLUMNS)
    got = got.reshape(len(L), 3, na).transpose(0, 2, 1)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


def test_passes(case):
    """A buffer of a few columns: several passes of one width and a rest."""
    ctx, b, L = case
    rng = np.random.default_rng(7)
    na = 400
    C, D = rng.normal(size=(b.nao, na)), rng.normal(size=(b.nao, 2))
    ref = np.matmul(np.matmul(C.T, L), D)
    got = ctx.mo_transform(C, 1, na, D, 1, 2, max_buffer_mb=max(1, 8 * len(L) * b.nao * 90 // 2 ** 20),
                           flags=lib.MO_ALL_COLUMNS)
    got = got.reshape(len(L), 2, na).transpose(0, 2, 1)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
