"""Connected components where their trees are deepest: every voxel solid, long rods and
serpentines, and blocks whose parts meet in faces, edges or corners only.  The mesh is
compared with the oracle's, entry by entry."""
import numpy as np
import pytest

from helpers import random_mask

pytestmark = pytest.mark.gpu


def _serpentine(n):
    """One path through every second row and layer, turned at alternate ends."""
    phi = np.zeros((n, n, n), np.int8)
    for z in range(0, n, 2):
        for y in range(0, n, 2):
            phi[z, y] = 1
            if y + 2 < n:
                phi[z, y + 1, -1 if y % 4 == 0 else 0] = 1
        if z + 2 < n:
            phi[z + 1, -1 if z % 4 == 0 else 0, 0] = 1
    return phi


def _checker(n):
    z, y, x = np.indices((n, n, n))
    return ((x + y + z) % 2).astype(np.int8)


def _islands(n):
    phi = np.zeros((n, n, n), np.int8)
    phi[0] = 1
    phi[3:6, 3:6, 3:6] = 1
    phi[6, 6, 6] = 1                       # hangs on a corner
    phi[2:4, n - 4, 2] = 1
    phi[n - 3, 2:n - 2, n - 3] = 1
    return phi


CASES = {
    "one voxel": lambda: np.ones((1, 1, 1), np.int8),
    "rod in x": lambda: np.ones((1, 1, 300), np.int8),
    "rod in z": lambda: np.ones((300, 1, 1), np.int8),
    "solid 33": lambda: np.ones((33, 33, 33), np.int8),
    "serpentine 17": lambda: _serpentine(17),
    "checker 12": lambda: _checker(12),
    "islands 11": lambda: _islands(11),
    "sparse": lambda: random_mask((19, 23, 29), 0.12, 7),
    "dense": lambda: random_mask((17, 16, 18), 0.8, 8),
}


@pytest.mark.parametrize("nen", [8, 20])
@pytest.mark.parametrize("name", list(CASES))
def test_mesh_equals_the_oracle(name, nen):
    import dtc_amd as dtc
    from oracle import oracle as O
    phi = CASES[name]()
    nodes, elems = dtc.mesh(phi, 1, nen, (0.01,) * 3, (2, 2, 2))
    onodes, oelems = O.mesh(phi, 1, nen, (0.01,) * 3, (2, 2, 2))
    assert np.array_equal(elems, oelems) and np.array_equal(nodes, onodes)


def test_solid_100_keeps_every_element_and_node():
    """The widest concurrent shortcutting: 10^6 voxels of one component."""
    import dtc_amd as dtc
    for _ in range(3):
        assert dtc.mesh_count(np.ones((100, 100, 100), np.int32), 1, 8) == (100 ** 3, 101 ** 3)
