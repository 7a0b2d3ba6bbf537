"""Edges of the Hermite potential kernels behind gi_coulomb_energy_grad:
numbers of primitive pairs around the 64 lanes of a tile and the four slices
of a workgroup, one pair alone, contracted pairs (several primitive pairs a
shell pair), every bra and ket order up to f pairs, and bases whose highest
pairs (g, h) leave the kernels for the row-sum path.  Energy and gradient
against the oracle; the bars are those of the other gradient tests: an energy
is a sum of terms exact to about 1e-14 of the largest (1e-12 of the sum), a
gradient component to 1e-8 (the oracle's own route)."""
import numpy as np
import pytest

import pyoracle
from gigpu import lib
from gigpu.basis import build_basis
from grad_helpers import random_density

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    pyoracle.build()
    c = lib.Context(0)
    yield c
    c.close()


def _check(ctx, b, seed, kappa=0.0, grad=True):
    D = random_density(b.nao, seed=seed)
    ctx.set_basis(b)
    o = pyoracle.Oracle(b)
    ref = o.coulomb_energy(D, kappa)
    e = ctx.coulomb_energy(D, kappa, grad=False)
    assert abs(e - ref) <= 1e-12 * max(1.0, abs(ref))
    if grad:
        e2, g = ctx.coulomb_energy(D, kappa)
        assert abs(e2 - ref) <= 1e-12 * max(1.0, abs(ref))
        gr = o.coulomb_grad(D, kappa=kappa)
        assert np.abs(g - gr).max() <= 1e-8 * max(1.0, np.abs(gr).max())


# n s shells have n (n + 1) / 2 pairs: 1, 55, 66, 120, 136, 253
@pytest.mark.parametrize("n", [1, 10, 11, 15, 16, 22])
@pytest.mark.parametrize("kappa", [0.0, 0.7])
def test_pair_counts(ctx, n, kappa):
    rng = np.random.default_rng(n)
    shells = {"H": [(0, [float(a)], [1.0]) for a in np.geomspace(0.2, 30.0, n)]}
    b = build_basis(["H"], rng.uniform(-1.0, 1.0, (1, 3)), shells)
    _check(ctx, b, n, kappa)


@pytest.mark.parametrize("lmax", [1, 2, 3])
def test_far_and_contracted(ctx, lmax):
    """Two atoms 60 bohr apart (every cross argument in the asymptotic range of
    the Boys function) and one near, contracted and single shells of every l."""
    O = [(l, [3.0, 0.9, 0.4], [0.3, 0.5, 0.4]) for l in range(lmax + 1)]
    H = [(l, [0.7], [1.0]) for l in range(lmax + 1)]
    xyz = np.array([[0.0, 0.0, 0.0], [1.1, 0.4, -0.3], [35.0, -40.0, 28.0]])
    _check(ctx, build_basis(["O", "H", "H"], xyz, {"O": O, "H": H}), 30 + lmax)


@pytest.mark.parametrize("top,grad", [(4, True), (5, False)])
def test_beyond_the_kernels(ctx, top, grad):
    O = [(0, [0.5], [1.0]), (2, [0.9], [1.0]), (top, [0.8], [1.0])]
    H = [(0, [0.4, 1.3], [0.6, 0.5]), (1, [0.6], [1.0]), (3, [1.1], [1.0])]
    xyz = np.array([[0.0, 0.2, -0.1], [1.3, 0.9, 0.4]])
    _check(ctx, build_basis(["O", "H"], xyz, {"O": O, "H": H}), 40 + top, grad=grad)
