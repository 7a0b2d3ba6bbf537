"""Primitive steps of contracted pairs through tiles of several bra pairs.

The 4x4x4 kernels evaluate the Boys values of consecutive (bra pair, bra
primitive, ket primitive) steps in one pass.  Small requests make tiles of one
bra pair; with the tile target at zero every tile takes four, of different
numbers of primitives, and the passes begin and end inside and across pairs.
ERIs to 1e-12 absolute, the bound of the other ERI tests."""
import numpy as np
import pytest

from gigpu.basis import build_basis

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _basis(seed):
    rng = np.random.default_rng(seed)

    def shell(l, n, a0):
        return (l, [a0 * 2.7 ** k for k in range(n)][::-1], list(rng.uniform(0.2, 0.8, n)))
    shells = {"O": [shell(0, 4, 0.15), shell(0, 1, 0.3), shell(1, 3, 0.2), shell(2, 2, 0.3), shell(2, 1, 0.7),
                    shell(3, 2, 0.6)],
              "H": [shell(0, 3, 0.1), shell(1, 1, 0.5)]}
    coords = np.array([[0.0, 0.0, 0.0], [1.43, 1.1, 0.0], [-1.43, 1.1, 0.2]])
    return build_basis(["O", "H", "H"], coords, shells, spher_ao=True)


@pytest.mark.parametrize("tiles", [0, 2048], ids=["four-bra-pairs", "one-bra-pair"])
def test_steps_across_bra_pairs(gpu_ctx, oracle_mod, tiles):
    b = _basis(23)
    o = oracle_mod.Oracle(b)
    gpu_ctx.set_basis(b)
    ns = b.nshells
    allp = [(A, B) for A in range(ns) for B in range(A + 1)]
    cp = allp[::2]
    try:
        gpu_ctx.set_option("eri_md4_tiles", tiles)
        V = gpu_ctx.eri_pair_block(allp, cp)
    finally:
        gpu_ctx.set_option("eri_md4_tiles", 2048)
    nang = b.shell_nang
    r0 = 0
    for (A, B) in allp:
        nr = nang(A) * nang(B)
        c0 = 0
        for (Cs, D) in cp:
            nc = nang(Cs) * nang(D)
            ref = o.eri(A, B, Cs, D).transpose(1, 0, 3, 2).reshape(nr, nc)
            assert np.abs(V[r0:r0 + nr, c0:c0 + nc] - ref).max() <= TOL, (A, B, Cs, D)
            c0 += nc
        r0 += nr
