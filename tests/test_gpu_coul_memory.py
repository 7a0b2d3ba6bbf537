"""What a context holds after the Coulomb gradient: its device arrays stay for
the next call up to 1 GiB, and are freed at the end of a call that needed more."""
import ctypes as C

import numpy as np
import pytest
import torch

from gigpu import lib, systems

pytestmark = pytest.mark.gpu


def _pool_bytes():
    """Bytes in use of the device's stream-ordered memory pool."""
    hip = C.CDLL("libamdhip64.so")
    pool, used = C.c_void_p(), C.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, 7, C.byref(used)) == 0   # hipMemPoolAttrUsedMemCurrent
    return used.value


@pytest.mark.parametrize("waters,freed", [(2, False), (6, True)])   # 0.37 and 1.2 GiB of arrays
def test_arrays_after_a_call(waters, freed):
    b = systems.water_system(waters, 6.0 * max(1.0, waters / 4.0) ** (1.0 / 3.0), "large", seed=3, contracted=True)
    D = systems.occupied_density(b.nao, 5 * waters, 3)
    c = lib.Context(0)
    try:
        c.set_basis(b)
        torch.cuda.synchronize()
        before = _pool_bytes()
        e, g = c.coulomb_energy(D)
        torch.cuda.synchronize()
        held = _pool_bytes() - before
        assert (held < 1 << 20) if freed else (1 << 20 < held <= 1 << 30)
        e2, g2 = c.coulomb_energy(D)   # on fresh arrays or the kept ones: the same sums
        assert e == e2 and np.array_equal(g, g2)
    finally:
        c.close()
