"""Particles across the host boundary: triples packed and unpacked on the
device, read back through the pinned ring.

Counts sit at the edges of a 256-particle workgroup, of the smallest staged
copy (256 KiB), of a 2 MiB ring chunk, of the size that starts copy threads
(8 MiB) and past the whole ring (32 MiB).  A freshly initialized scene gives
back what was loaded: bit for bit with the identity transform, and otherwise
what the float operations give in numpy.
"""

import threading

import numpy as np
import pytest

import flipengine3d_amd as fa
from tests.helpers import bits_equal, dam, radius

pytestmark = pytest.mark.gpu


def _scene(gpu, n, seed, offset=None, scale=None):
    sim = fa.FluidSimulation(16, 12, 20, 1 / 16, ctx=gpu)
    if offset is not None:
        sim.setDomainOffset(*offset)
        sim.setDomainScale(scale)
    rng = np.random.default_rng(seed)
    grid = (rng.random((n, 3)) * np.array([15.9, 11.9, 19.9]) / 16).astype(np.float32)
    pos = grid if offset is None else grid * np.float32(scale) + np.array(offset, np.float32)
    vel = rng.standard_normal((n, 3)).astype(np.float32)
    sim.loadMarkerParticleData(pos, vel)
    sim.initialize()
    return sim, pos, vel


@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 21845, 21846, 174762, 174763, 699050, 699051, 2900000])
def test_read_back_is_what_was_loaded(gpu, n):
    sim, pos, vel = _scene(gpu, n, seed=n)
    p, v = sim.particles()
    assert bits_equal(p, pos) and bits_equal(v, vel)
    if n > 300:
        for a, b in ((0, 1), (7, n - 3), (n - 257, n)):
            p, v = sim.particles_range(a, b)
            assert bits_equal(p, pos[a:b]) and bits_equal(v, vel[a:b])
    sim.close()


def test_domain_transform_is_float_arithmetic(gpu):
    off, scale = (0.3, -1.7, 2.5), 1.3
    sim, pos, vel = _scene(gpu, 5000, 3, off, scale)
    inv = np.float32(1.0 / np.float64(np.float32(scale)))
    grid = (pos - np.array(off, np.float32)) * inv
    hi = np.array([16, 12, 20]) / 16
    keep = ((grid >= 0) & (grid.astype(np.float64) < hi)).all(1)
    p, v = sim.particles()
    assert bits_equal(p, grid[keep] * np.float32(scale) + np.array(off, np.float32))
    assert bits_equal(v, vel[keep])
    sim.close()


def test_threads_share_the_staging(gpu):
    scenes = [_scene(gpu, 400000 + 1000 * q, seed=q) for q in range(4)]
    bad = []

    def read(q):
        sim, pos, vel = scenes[q]
        for _ in range(5):
            p, v = sim.particles()
            if not (bits_equal(p, pos) and bits_equal(v, vel)):
                bad.append(q)

    threads = [threading.Thread(target=read, args=(q,)) for q in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_stage_calls_share_the_pool(gpu, oracle):
    # Two contexts, calls of different sizes in turn and from two threads:
    # blocks given back by one call are another's.
    other = fa.Context(0)
    cases = []
    for dims in ((20, 18, 22), (40, 33, 30), (16, 16, 16)):
        s = dam(*dims, seed=4)
        cases.append((dims, s, oracle.liquid_sdf(*dims, s.dx, s.positions, radius(s.dx))))
    bad = []

    def call(ctx):
        for _ in range(6):
            for dims, s, want in cases:
                if not bits_equal(ctx.liquid_sdf(*dims, s.dx, s.positions, radius(s.dx)), want):
                    bad.append(dims)

    threads = [threading.Thread(target=call, args=(c,)) for c in (gpu, other)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
