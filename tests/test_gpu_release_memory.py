"""Device memory that the library keeps for its next calls goes back to the program."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free_bytes():
    from dtc_amd._lib import load
    free, total = C.c_size_t(), C.c_size_t()
    assert load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # the library's own runtime
    return free.value


def test_kept_memory_is_given_back():
    """The mesher's work space of blocks of 96^3 to 160^3 voxels (over 256 MiB kept, 26 bytes a
    half-voxel lattice node and more) is free again after the release, but for what the
    runtime rounds up (64 MiB)."""
    import dtc_amd as dtc
    dtc.release_memory()
    free0 = _free_bytes()
    for n in (96, 128, 160):
        phi = np.zeros((n, n, n), np.int32)
        phi[:2] = 1
        dtc.mesh(phi, 1, 20, (0.01,) * 3, (2, 2, 2))
    assert free0 - _free_bytes() > (256 << 20)
    dtc.release_memory()
    assert free0 - _free_bytes() <= (64 << 20)


def test_a_live_batch_keeps_its_memory():
    import dtc_amd as dtc
    from dtc_amd import synth
    doms = [dtc.Domain(synth.trabecular(14 + i, seed=i, sigma=1.5, bvtv=0.4), delta=(0.01,) * 3) for i in range(3)]
    with dtc.Batch(doms, precision=1, precond=1, rotation=False) as b:
        first = b.run()
        g0 = b.grad(1, np.eye(6))
        dtc.release_memory()
        g1 = b.grad(1, np.eye(6))
        again = b.run()
    assert np.array_equal(g0, g1)
    for x, y in zip(first, again):
        assert x["status"] == y["status"] == 0 and np.array_equal(x["ff"], y["ff"])
