"""Velocity extrapolation against the oracle, bit for bit, where its four faces
a thread can go wrong: face counts of every remainder, rows shorter than a
word, grids without an interior, valid faces next to the border and none at
all, and more layers than the grid has."""
import numpy as np
import pytest

from tests.helpers import bits_equal

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (2, 3, 1), (3, 3, 3), (3, 5, 3), (4, 4, 4), (5, 4, 7), (6, 3, 9), (7, 7, 7), (33, 5, 4), (34, 18, 3),
        (67, 9, 21)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("share", [0.0, 0.02, 0.6])
def test_random_masks(gpu, oracle, dims, share):
    rng = np.random.default_rng(dims[0] * 100 + dims[1])
    shape = dims[::-1]
    grid = rng.standard_normal(shape).astype(np.float32)
    valid = (rng.random(shape) < share).astype(np.uint8)
    for layers in (0, 1, 2, 7, 250):
        assert bits_equal(gpu.extrapolate(grid, valid, layers), oracle.extrapolate(grid, valid, layers))
