"""The mixed-precision solve's multigrid preconditioner where it can go wrong.

Level sizes: bricks are 64 x 2 x 2 cells, levels halve with an odd cell left
over, levels of up to 2048 cells are done by one workgroup; the grids below
leave remainders on every axis, have one to three levels above that workgroup
and, the smallest, a single cell per level.  Both paths stop on the same FP64
true residual, 1e-9 of |b|_inf, so the pressures agree to the bound the mixed
path states (1e-6 of the largest) and the velocities to 1e-5 of the fastest.

What it does not solve goes to the MIC(0) iteration, which treats the system
as the FP64 path does: an iteration cap below its need, values that are not
finite.  So does, in the projection call, a pocket that borders no air (its
pressure is fixed up to a constant, which follows from the preconditioner).
"""

import numpy as np
import pytest

from tests.helpers import bits_equal, dam, pocket_inputs
from tests.test_gpu_mixed import _projection_inputs

pytestmark = pytest.mark.gpu

FP64, MIXED = 0, 1


def _both(gpu, inputs, dims, **kw):
    dx, _, weights, liquid, mac, valid = inputs
    return [gpu.pressure_solve(*dims, dx, 1 / 60, liquid, weights, mac, valid, precision=p, **kw)
            for p in (FP64, MIXED)]


@pytest.mark.parametrize("dims", [(8, 5, 6), (66, 9, 7), (67, 35, 34), (131, 20, 18), (30, 67, 26), (90, 70, 74)])
@pytest.mark.parametrize("box", [(0.0, 0.0, 0.0, 0.45, 0.6, 1.0), (0.3, 0.0, 0.1, 1.0, 0.55, 0.9)])
def test_level_sizes(gpu, oracle, dims, box):
    inputs = _projection_inputs(oracle, *dims, seed=5, box=box)
    a, b = _both(gpu, inputs, dims)
    assert a["ok"] == b["ok"] == 1 and a["rows"] == b["rows"] > 0
    # One true residual confirms a multigrid solve.  The smallest grid's single
    # layer touches no air in one of the boxes.
    assert b["refinements"] == 1 or dims == (8, 5, 6)
    assert np.abs(a["soln"] - b["soln"]).max() <= 1e-6 * np.abs(a["soln"]).max()
    vmax = max(float(np.abs(g).max()) for g in a["mac"])
    for x, y in zip(a["mac"], b["mac"]):
        assert np.abs(x.astype(np.float64) - y).max() <= 1e-5 * vmax
    for x, y in zip(a["valid"], b["valid"]):
        assert bits_equal(x, y)


def test_no_rows(gpu, oracle):
    for dims in ((2, 5, 5), (3, 3, 3)):
        z = [np.zeros(s, np.float32) for s in ((dims[2], dims[1], dims[0] + 1), (dims[2], dims[1] + 1, dims[0]),
                                               (dims[2] + 1, dims[1], dims[0]))]
        phi = np.ones(dims[::-1], np.float32)
        valid = [np.zeros(g.shape, np.uint8) for g in z]
        for p in (FP64, MIXED):
            r = gpu.pressure_solve(*dims, 0.1, 0.01, phi, (*z, np.zeros_like(phi)), z, valid, precision=p)
            assert r["ok"] == 1 and r["rows"] == 0 and r["iters"] == 0


@pytest.mark.parametrize("cap", [1, 4])
def test_capped_solve_is_mic0s(gpu, oracle, cap):
    # As many iterations of the same method in FP32 and in FP64: the iterates
    # agree to FP32 rounding.
    dims = (24, 28, 21)
    a, b = _both(gpu, _projection_inputs(oracle, *dims), dims, maxiter=cap)
    assert a["iters"] == b["iters"] == cap and a["ok"] == b["ok"]
    assert abs(a["err"] - b["err"]) <= 1e-5 * a["err"]
    assert np.abs(a["soln"] - b["soln"]).max() <= 1e-5 * np.abs(a["soln"]).max()


def test_not_finite(gpu, oracle):
    dims = (24, 28, 21)
    inputs = list(_projection_inputs(oracle, *dims))
    bad = [g.copy() for g in inputs[4]]
    bad[0][10, 8, 5] = np.nan
    a, b = _both(gpu, [*inputs[:4], bad, inputs[5]], dims)
    assert a["ok"] == b["ok"] == 0
    for x, y in zip(a["mac"], b["mac"]):
        assert bits_equal(x, y)
    a, b = _both(gpu, inputs, dims)
    assert a["ok"] == b["ok"] == 1


def test_not_finite_in_a_field_at_rest(gpu, oracle):
    # Every other row of the right-hand side is zero.
    dims = (24, 28, 21)
    dx, solid, weights, liquid, mac, valid = _projection_inputs(oracle, *dims)
    still = [np.zeros_like(g) for g in mac]
    rows = (liquid < 0) & (weights[1][:, 1:] > 0)
    k, j, i = np.argwhere(rows[1:-1, 1:-1, 1:-1])[5] + 1
    still[1][k, j + 1, i] = np.nan
    a, b = _both(gpu, (dx, solid, weights, liquid, still, valid), dims)
    assert a["ok"] == b["ok"] == 0
    for x, y in zip(a["mac"], b["mac"]):
        assert bits_equal(x, y)


def test_pocket_keeps_its_constant(gpu, oracle):
    dims = (20, 18, 17)
    dx, solid, weights, liquid, mac, valid, *_ = pocket_inputs(oracle, *dims)
    a, b = _both(gpu, (dx, solid, weights, liquid, mac, valid), dims)
    assert a["ok"] == b["ok"] == 1
    assert np.abs(a["soln"] - b["soln"]).max() <= 1e-6 * np.abs(a["soln"]).max()


def test_scene_goes_on_after_mic0_took_over(gpu):
    # The smallest scenes that solve with multigrid hold 2^20 cells.
    import flipengine3d_amd as fa
    I, J, K = 1024, 32, 32
    s = dam(I, J, K, seed=2, box=(0.0, 0.0, 0.0, 0.2, 0.5, 1.0))
    sims = []
    for prec in (fa.PCG_FP64, fa.PCG_MIXED):
        sim = fa.FluidSimulation(I, J, K, s.dx, ctx=gpu, precision=prec)
        sim.addBodyForce(0.0, -9.81, 0.0)
        sim.setPressureSolverTolerance(1e-9, 5)
        sim.loadMarkerParticleData(s.positions, s.velocities)
        sim.initialize()
        sim.set_launch_graphs(True)
        sims.append(sim)
    for f in range(3):
        st = [sim.update(1 / 480) for sim in sims]
        assert st[0].pressure_ok == st[1].pressure_ok and st[0].pcg_iterations == st[1].pcg_iterations
        (p0, v0), (p1, v1) = sims[0].particles(), sims[1].particles()
        assert np.abs(p0 - p1).max() <= 1e-3 * s.dx and np.abs(v0 - v1).max() <= 1e-3


def test_scene_on_either_side_of_the_line(gpu):
    # 2^20 cells and one plane less: both follow the FP64 path.
    import flipengine3d_amd as fa
    for I in (1024, 1023):
        s = dam(I, 32, 32, seed=3, box=(0.0, 0.0, 0.0, 0.15, 0.6, 1.0))
        sims = []
        for prec in (fa.PCG_FP64, fa.PCG_MIXED):
            sim = fa.FluidSimulation(I, 32, 32, s.dx, ctx=gpu, precision=prec)
            sim.addBodyForce(0.0, -9.81, 0.0)
            sim.loadMarkerParticleData(s.positions, s.velocities)
            sim.initialize()
            sim.set_launch_graphs(True)
            sims.append(sim)
        for _ in range(2):
            st = [sim.update(1 / 480) for sim in sims]
            assert st[0].pressure_ok == st[1].pressure_ok == 1
            # Multigrid confirms with one true residual; MIC(0) in FP32 replaces
            # its residual several times on the way.
            assert (st[1].pcg_refinements == 1) == (I == 1024)
        (p0, v0), (p1, v1) = sims[0].particles(), sims[1].particles()
        assert p0.shape == p1.shape
        assert np.abs(p0 - p1).max() <= 1e-3 * s.dx and np.abs(v0 - v1).max() <= 1e-3


def test_graph_batches_match_kernel_launches(gpu):
    import flipengine3d_amd as fa
    s = dam(1024, 32, 32, seed=7, box=(0.0, 0.0, 0.0, 0.12, 0.5, 1.0))
    sims = []
    for graphs in (False, True):
        sim = fa.FluidSimulation(1024, 32, 32, s.dx, ctx=gpu, precision=fa.PCG_MIXED)
        sim.addBodyForce(0.0, -9.81, 0.0)
        sim.loadMarkerParticleData(s.positions, s.velocities)
        sim.initialize()
        sim.set_launch_graphs(graphs)
        sims.append(sim)
    for _ in range(4):
        st = [sim.update(1 / 480) for sim in sims]
        assert st[0].pcg_iterations == st[1].pcg_iterations and st[0].pressure_ok == st[1].pressure_ok == 1
        for x, y in zip(sims[0].particles(), sims[1].particles()):
            assert bits_equal(x, y)


def _closed_region(liquid, weights, start):
    """Cells of the liquid region of `start` over open faces, and whether one of those faces leads to air."""
    wu, wv, ww = weights
    cells, todo, air = {start}, [start], False
    while todo:
        k, j, i = todo.pop()
        for w, n in ((wu[k, j, i + 1], (k, j, i + 1)), (wu[k, j, i], (k, j, i - 1)), (wv[k, j + 1, i], (k, j + 1, i)),
                     (wv[k, j, i], (k, j - 1, i)), (ww[k + 1, j, i], (k + 1, j, i)), (ww[k, j, i], (k - 1, j, i))):
            if w <= 0:
                continue
            if liquid[n] >= 0:
                air = True
            elif n not in cells:
                cells.add(n)
                todo.append(n)
    return cells, air


def test_closed_cavity_in_a_scene(gpu):
    # A cavity full of liquid between six slabs borders no air: multigrid solves
    # it with the rest, and the velocities follow the FP64 path's.
    import flipengine3d_amd as fa
    from flipengine3d_amd import scenes
    I, J, K, dx = 1024, 32, 32, 1 / 32
    lo, hi = np.array([600.4, 8.4, 9.4]), np.array([608.7, 16.7, 17.7])  # cavity, in cells
    rng = np.random.default_rng(5)
    cells = np.stack(np.meshgrid(np.arange(2, 120), np.arange(2, 16), np.arange(2, 30), indexing="ij"), -1).reshape(-1, 3)
    inner = np.stack(np.meshgrid(*[np.arange(int(a), int(b) + 1) for a, b in zip(lo, hi)], indexing="ij"), -1)
    cells = np.concatenate([cells, inner.reshape(-1, 3)])
    off = np.array([[a, b, c] for a in (0.25, 0.75) for b in (0.25, 0.75) for c in (0.25, 0.75)])
    p = (cells[:, None] + off[None]).reshape(-1, 3)
    p += (rng.random(p.shape) - 0.5) * 0.2
    in_cavity = ((p > lo + 0.05) & (p < hi - 0.05)).all(1)
    p = p[(p[:, 0] < 200) | in_cavity]
    pos = (p * dx).astype(np.float32)
    vel = (0.3 * rng.standard_normal(pos.shape)).astype(np.float32)
    sims = []
    for prec in (fa.PCG_FP64, fa.PCG_MIXED):
        sim = fa.FluidSimulation(I, J, K, dx, ctx=gpu, precision=prec)
        sim.addBodyForce(0.0, -9.81, 0.0)
        sim.setMinTimeStepsPerFrame(1)
        sim.setMaxTimeStepsPerFrame(1)
        for a in range(3):
            for side in (0, 1):
                b0, b1 = lo - 3, hi + 3
                if side:
                    b0[a] = hi[a]
                else:
                    b1[a] = lo[a]
                sim.addMeshObstacle(*scenes.box_mesh(b0 * dx, b1 * dx))
        sim.loadMarkerParticleData(pos, vel)
        sim.initialize()
        sims.append(sim)
    for step in range(2):
        st = [sim.update(1 / 480) for sim in sims]
        if step == 0:
            region, air = _closed_region(sims[1].grid(0), [sims[1].grid(w) for w in (5, 6, 7)], (13, 12, 604))
            assert len(region) >= 7 ** 3 and not air
        assert st[0].pressure_ok == st[1].pressure_ok == 1
        assert st[1].pcg_refinements == 1 and st[1].pcg_iterations <= 40  # multigrid's
        (p0, v0), (p1, v1) = sims[0].particles(), sims[1].particles()
        assert p0.shape == p1.shape
        assert np.abs(p0 - p1).max() <= 1e-3 * dx and np.abs(v0 - v1).max() <= 1e-3
