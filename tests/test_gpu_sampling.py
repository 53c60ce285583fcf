"""Velocity sampling and advection against the oracle, bit for bit, where the
cells of the three components reach the edge of their grids: on the walls, half
a cell from them, just inside and outside them, on grids down to one cell."""
import itertools

import numpy as np
import pytest

from tests.helpers import bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 3), (3, 2, 2), (5, 4, 3)])
def test_at_the_edges_of_the_grids(gpu, oracle, dims):
    rng = np.random.default_rng(sum(dims))
    I, J, K = dims
    dx = 0.125
    mac = [rng.standard_normal(s).astype(np.float32) for s in ((K, J, I + 1), (K, J + 1, I), (K + 1, J, I))]
    marks = []
    for n in dims:
        hi = np.float32(n * dx)
        marks.append([0.0, -1e-3, 0.5 * dx, hi, hi - 0.5 * dx, np.nextafter(hi, np.float32(0)), 0.5 * hi, 1.5 * hi])
    pos = np.array(list(itertools.product(*marks)), np.float32)
    pos = np.concatenate([pos, (rng.random((200, 3)) * (np.array(dims) + 1) * dx - 0.5 * dx).astype(np.float32)])
    assert bits_equal(gpu.trilinear_velocity(I, J, K, dx, mac, pos), oracle.trilinear_velocity(I, J, K, dx, mac, pos))
    for order in (1, 2, 3, 4):
        assert bits_equal(gpu.advect_particles(I, J, K, dx, mac, pos, 0.02, order),
                          oracle.advect_particles(I, J, K, dx, mac, pos, 0.02, order))
