"""The surface field by nodes and by particles against the oracle, bit for bit,
on both sides of the line between them: kernels whose reach ends before, at and
past the half-cells a node looks at, one to three nodes a cell, ragged grids,
and particles thinned out until most nodes lie in the outer bands."""
import numpy as np
import pytest

from tests.helpers import bits_equal, dam

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sub", [1, 2, 3])
@pytest.mark.parametrize("scale", [1.5, 3.0, 3.15, 3.3, 4.5])
def test_both_sides_of_the_line(gpu, oracle, sub, scale):
    I, J, K = 21, 17, 19
    s = dam(I, J, K, seed=5, box=(0.0, 0.0, 0.0, 0.6, 0.7, 1.0))
    solid, _ = oracle.domain_solid(I, J, K, s.dx)
    rng = np.random.default_rng(7)
    for share in (1.0, 0.05):
        pos = s.positions[rng.random(len(s.positions)) < share]
        ref = oracle.surface_mesh(I, J, K, s.dx, pos, solid, subdivisions=sub, particle_scale=scale)
        got = gpu.mesh_particles(I, J, K, s.dx, pos, solid, subdivisions=sub, particle_scale=scale)
        assert ref[0].shape == got[0].shape and bits_equal(got[0], ref[0])
        assert np.array_equal(got[1], ref[1])
