"""Products on the int8 matrix cores (crt.hip) in several slices of the larger
operand and chunks of k: the vectors Inv_L V(P, pq) with slices of columns, or,
for a decomposition with more vectors than columns in a subset, slices of rows
of the triangular Inv_L; and what the context holds of their work arrays.

The bar is the scheme's own, as in test_gpu_crt.py: half a unit an element at
row norms of 2^57..2^58 units, sqrt(k) 2^-57 |a| |b|, plus one rounding of the
result and the reference's own."""
import ctypes as C

import numpy as np
import pytest
import torch

from gigpu import lib, systems

pytestmark = pytest.mark.gpu


class _Device:
    def __init__(self, pointer, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (pointer, False), "strides": None,
                                         "version": 2}


def _check_vectors(c, b):
    """Sampled elements of Rkpq, rows from every tile column of 256, against extended precision."""
    m, X = c.chol_meta(), c.chol_inv_l()
    nv, msd = m["nvecs"], m["max_subset_dim"]
    R = torch.as_tensor(_Device(c.chol_rkpq_device_ptr(), (m["nsubsets"], msd, nv)), device="cuda")
    sp, loc = m["shell_pairs"], m["shell_pair_loc"]
    piv = [tuple(sp[i - 1] - 1) for i in m["pivot_shell_pairs"]]
    sel, off, k = [], 0, 0
    for (p, q), n in zip(piv, m["pivot_shell_pair_dim"]):
        sel += [off + m["pivot_orb_pairs"][k + j] - 1 for j in range(n)]
        k += n
        off += b.shell_nang(p) * b.shell_nang(q)
    rng = np.random.default_rng(7)
    pick = [s for s in [0, 1, len(sp) - 2, len(sp) - 1] + list(rng.choice(len(sp), 8, replace=False))
            if sp[s][0] != sp[s][1]]
    V = c.eri_pair_block([tuple(sp[s] - 1) for s in pick], piv)[:, sel]
    rows = np.unique(np.concatenate([np.arange(0, nv, 256), np.arange(255, nv, 256), [nv - 1]]))
    at = torch.from_numpy(rows).cuda()
    got = np.concatenate([R[loc[s][2] - 1, loc[s][1] - 1:loc[s][1] - 1 + m["shell_pair_dim"][s]][:, at].cpu().numpy()
                          for s in pick]).T
    A = X[rows]
    ref = np.asarray(A, np.longdouble) @ np.asarray(V, np.longdouble).T
    bar = (np.sqrt(nv) * 2.0 ** -57 * np.linalg.norm(A, axis=1)[:, None] * np.linalg.norm(V, axis=1)[None, :]
           + 2.0 ** -52 * np.abs(ref) + np.sqrt(nv) * 2.0 ** -63 * (np.abs(A) @ np.abs(V).T)).astype(float)
    err = np.abs(got - ref).astype(float)
    assert (err <= bar).all(), (float((err / bar).max()), rows[(err > bar).any(axis=1)][:8])


def test_triangular_rows_in_slices():
    b = systems.water_system(6, 7.2, "large", seed=41)
    c = lib.Context(0)
    try:
        c.set_basis(b)
        c.set_option("vec_stage_mb", 1)   # a product for every subset of at most 4003 columns
        c.set_option("int8_work_mb", 1)   # slices of 2048 rows, the smallest
        c.chol_build(tau=1e-10)
        d = c.chol_dims()
        # more rows than columns, in three slices; the int8 route is the faster one from 4800 x 3600 on
        assert d["nvecs"] > 4800 and d["nvecs"] % 256 != 0 and 3600 < d["max_subset_dim"] < d["nvecs"]
        _check_vectors(c, b)
    finally:
        c.close()


@pytest.mark.parametrize("stage_mb,work_mb", [
    (1, 1140),      # subset by subset, all of k at once: three slices of rows
    (16384, 1140),  # all subsets at once, all of k at once: slices of 2048 columns
    (16384, 1),     # and three chunks of k, the smallest
])
def test_slices_and_chunks(stage_mb, work_mb):
    b = systems.water_system(6, 7.2, "large", seed=41)
    c = lib.Context(0)
    try:
        c.set_basis(b)
        c.set_option("int8_work_mb", 0)   # DGEMM
        c.chol_build(tau=1e-10)
        ref = c.chol_meta()
        c.set_option("vec_stage_mb", stage_mb)
        c.set_option("int8_work_mb", work_mb)
        c.chol_build(tau=1e-10)
        m = c.chol_meta()
        # SubtractR goes the same ways (more rows than columns, added to M): the same pivots
        assert m["nvecs"] == ref["nvecs"] > 4800
        assert (m["pivot_order"] == ref["pivot_order"]).all()
        _check_vectors(c, b)
    finally:
        c.close()


def _pool_bytes():
    """Bytes in use of the device's stream-ordered memory pool."""
    hip = C.CDLL("libamdhip64.so")
    pool, used = C.c_void_p(), C.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, 7, C.byref(used)) == 0   # hipMemPoolAttrUsedMemCurrent
    return used.value


def test_work_arrays_are_given_back():
    """The int8 products' arrays go when the option is set, and with 0 a build
    allocates none of them."""
    b = systems.water_system(6, 7.2, "large", seed=41)
    c = lib.Context(0)
    try:
        c.set_basis(b)
        c.chol_build(tau=1e-5)
        torch.cuda.synchronize()
        held = _pool_bytes()
        c.set_option("int8_work_mb", 0)
        torch.cuda.synchronize()
        freed = _pool_bytes()
        # Inv_L's residues alone: 15 bytes an element of 2304 x 2304 at least
        assert c.chol_dims()["nvecs"] > 2048 and held - freed >= 15 * 2304 * 2304
        c.chol_build(tau=1e-5)
        torch.cuda.synchronize()
        assert _pool_bytes() == freed
    finally:
        c.close()


@pytest.mark.parametrize("work_mb", [9216, 64])   # four chunks of k; some thirty, with slices of vectors
def test_pair_products_of_orthonormal_points(work_mb):
    """XR = 2 Xgpq R^T itself: with orthonormal rows of X the metric is the
    identity (off its diagonal the squares of rounding errors), so Z = XR up to
    the rounding of S(g, g), some nao units of 2^-52."""
    b = systems.water_system(11, 8.8, "large", seed=5)
    c = lib.Context(0)
    try:
        c.set_basis(b)
        c.chol_build(tau=1e-5)
        c.set_option("int8_work_mb", work_mb)
        m = c.chol_meta()
        nv, msd = m["nvecs"], m["max_subset_dim"]
        n = 768   # three tiles of points: the int8 route is the faster one from some 3500 vectors on
        assert nv > 3800
        rng = np.random.default_rng(6)
        X = np.asfortranarray(np.linalg.qr(rng.standard_normal((b.nao, n)))[0].T)
        Z, _ = c.thc_z(X)
        k = np.unique(np.concatenate([[0, 255, 256, nv - 1], rng.choice(nv, 16, replace=False)]))
        R = torch.as_tensor(_Device(c.chol_rkpq_device_ptr(), (m["nsubsets"], msd, nv)), device="cuda")
        R = R[:, :, torch.from_numpy(k).cuda()].cpu().numpy()
    finally:
        c.close()
    loc0 = np.concatenate([[0], np.cumsum([b.shell_nang(s) for s in range(b.nshells)])])
    P, Q, cols = [], [], []
    for (A, B), (_, pos, sub) in zip(m["shell_pairs"], m["shell_pair_loc"]):
        na, nb = b.shell_nang(A - 1), b.shell_nang(B - 1)
        ab = [(i, j) for j in range(nb) for i in range(j if A == B else 0, na)]
        P += [loc0[A - 1] + i for i, _ in ab]
        Q += [loc0[B - 1] + j for _, j in ab]
        cols += [(sub - 1) * msd + pos - 1 + i for i in range(len(ab))]
    P, Q, V = np.array(P), np.array(Q), R.reshape(-1, len(k))[cols].T
    g = np.array([0, 1, 255, 256, 257, 511, 512, 700, n - 2, n - 1])
    A = X[np.ix_(g, P)] * X[np.ix_(g, Q)] * np.where(P == Q, 1.0, 2.0)
    ref = np.asarray(A, np.longdouble) @ np.asarray(V, np.longdouble).T
    ref /= (np.asarray(X[g], np.longdouble) ** 2).sum(1)[:, None] ** 2
    bar = (np.sqrt(len(P)) * 2.0 ** -57 * np.linalg.norm(A, axis=1)[:, None] * np.linalg.norm(V, axis=1)[None, :]
           + 4 * b.nao * 2.0 ** -52 * np.abs(ref)).astype(float)
    err = np.abs(Z[np.ix_(g, k)] - ref).astype(float)
    assert (err <= bar).all(), float((err / bar).max())
