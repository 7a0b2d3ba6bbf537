"""Split-BF16 MO transform at the edges of its 128 x 128 tiles and 256-k chunks
against the FP64 transform.  Bar: the slices of both operands are cut at 2^-32
of the largest element of a row's chunk, so with |C| <= 1 an element is off by
at most 2^-32 (2 nao) max|W|, W the half-transformed vectors, bounded here by
the FP64 transform with unit columns on the second side."""
import numpy as np
import pytest

from gigpu import lib, systems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 4])   # 75 and 300 AOs: below and above a chunk of k
def built(request):
    b = systems.water_system(request.param, 6.0, "large", seed=4)
    c = lib.Context(0)
    c.set_basis(b)
    c.chol_build(tau=1e-5)
    yield c, b
    c.close()


@pytest.mark.parametrize("na,nb", [(1, 1), (1, 65), (2, 64), (3, 31), (7, 66), (5, 70)])
def test_tiles(built, na, nb):
    c, b = built
    rng = np.random.default_rng(100 * na + nb)
    C, _ = np.linalg.qr(rng.normal(size=(b.nao, b.nao)))
    r64 = c.mo_transform(C, 1, na, C, na + 1, na + nb)
    r16 = c.mo_transform(C, 1, na, C, na + 1, na + nb, flags=lib.MO_SPLIT_BF16)
    W = c.mo_transform(C, 1, na, np.eye(b.nao), 1, b.nao)
    assert np.abs(r16 - r64).max() <= 2.0 ** -32 * 2 * b.nao * np.abs(W).max()


def test_wide(built):
    """More than one tile of columns where the basis has them."""
    c, b = built
    C, _ = np.linalg.qr(np.random.default_rng(5).normal(size=(b.nao, b.nao)))
    nb = b.nao - 3
    r64 = c.mo_transform(C, 1, 3, C, 4, 3 + nb)
    r16 = c.mo_transform(C, 1, 3, C, 4, 3 + nb, flags=lib.MO_SPLIT_BF16)
    W = c.mo_transform(C, 1, 3, np.eye(b.nao), 1, b.nao)
    assert np.abs(r16 - r64).max() <= 2.0 ** -32 * 2 * b.nao * np.abs(W).max()
