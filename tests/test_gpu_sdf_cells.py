"""The liquid SDF by cells (search radii under two cells) against the oracle.

The nearest particle is found in half-cells taken by distance, with skips and
reach tests that have to agree with the reference's block assignment and
index ranges to the bit: the field is compared bit for bit.  Cases: tile
remainders along each axis (16 x 4 x 4 cells), grids smaller than a tile,
sparse particles (every ring of half-cells is walked), particles on cell and
half-cell boundaries, radii up to the rule's limit and just past it, dense
cells, no particles, and a grid past 4096 cells along i, where every particle
in range is tested.
"""

import numpy as np
import pytest

from tests.helpers import bits_equal, ndiff, radius

pytestmark = pytest.mark.gpu


def _points(dims, dx, count, seed):
    I, J, K = dims
    rng = np.random.default_rng(seed)
    hi = np.array([I, J, K]) * dx
    pos = rng.random((count, 3)) * hi
    half = np.floor(rng.random((count // 4 + 1, 3)) * 2 * np.array([I, J, K])) * (0.5 * dx)
    pos = np.concatenate([pos, half]).astype(np.float32)
    return pos[((pos >= 0) & (pos.astype(np.float64) < hi)).all(1)]


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 3, 4), (16, 4, 4), (17, 5, 9), (33, 21, 12), (47, 30, 26),
                                  (4100, 4, 5)])
@pytest.mark.parametrize("per_cell", [0.0, 0.01, 0.3, 8.0])
def test_sdf_matches_oracle(gpu, oracle, dims, per_cell):
    I, J, K = dims
    dx = 1.0 / max(dims)
    pos = _points(dims, dx, int(per_cell * I * J * K) + 1, seed=I + 3 * J) if per_cell else np.zeros((0, 3), np.float32)
    for factor in (1.0, 0.4, 1.14):
        got = gpu.liquid_sdf(I, J, K, dx, pos, factor * radius(dx))
        want = oracle.liquid_sdf(I, J, K, dx, pos, factor * radius(dx))
        assert bits_equal(got, want), (dims, per_cell, factor, ndiff(got, want))


def test_sdf_dense_cells(gpu, oracle):
    I, J, K = 20, 13, 11
    dx = 1.0 / 20
    rng = np.random.default_rng(3)
    centre = np.array([7.3, 5.1, 4.9]) * dx
    pos = (centre + rng.normal(size=(6000, 3)) * 0.4 * dx).astype(np.float32)
    assert bits_equal(gpu.liquid_sdf(I, J, K, dx, pos, radius(dx)), oracle.liquid_sdf(I, J, K, dx, pos, radius(dx)))


def test_sdf_radius_past_the_rule(gpu, oracle):
    # 2 r >= 1.99 cells keeps the pass by particles, whose candidates end two
    # cells outside each 10^3 block: on one block it sees them all.
    I, J, K = 10, 9, 8
    dx = 0.1
    pos = _points((I, J, K), dx, 40, seed=9)
    for r in (0.994 * dx, 0.996 * dx, 1.3 * dx):
        got, want = gpu.liquid_sdf(I, J, K, dx, pos, r), oracle.liquid_sdf(I, J, K, dx, pos, r)
        assert bits_equal(got, want), (r, ndiff(got, want))
