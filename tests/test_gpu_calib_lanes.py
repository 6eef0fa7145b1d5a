"""The adjoint's reverse kernels give a sphere 16 or 32 lanes: a sphere count around a block's 8
and 16 spheres, one sphere, and the largest slot capacity (a lane for every history value). The
gradient of a weighted sum of the final positions agrees with central differences of the forward
run within 1e-3 of its size, the bound of the radial profile's gradient; the run is 40 steps of
touching spheres on a floor. The differences take the step 1e-8: contacts that nearly stick make
the forward run curved on the scale of 1e-6 in the parameters (17 spheres, d/d restitution, by
differences: 0.15617 at 1e-6, 0.10475 at 1e-7, 0.09957 at 1e-8; by the adjoint 0.09951), and the
rounding of positions of 0.1 leaves 1e-8 of the gradient's unit at this step.

The forward's contact kernel gives a wave 2 to 16 spheres by their number and its cell table 16^3
to 128^3 buckets, 128^3 whenever a sphere is larger than a cell: positions, velocities, Euler
parameters and rates are bit-identical with the oracle for every choice."""
import numpy as np
import pytest

import xdem_ref
from xdynamics_dll_amd import SceneData
from xdynamics_dll_amd.calib import Calibration

pytestmark = pytest.mark.gpu


def lattice(n, side=4):
    """n spheres row by row, side x side to a layer, each overlapping its neighbours and the floor by
    about 0.5 percent of a radius, moving."""
    scene = SceneData.build(5, 1005, np_override=n)
    rng = np.random.default_rng(n)
    r = 1.25e-3
    k = np.arange(n)
    cell = np.stack([k % side, k // side % side, k // side**2], axis=1)
    pos = np.empty((n, 4))
    pos[:, :3] = np.array([0.1, 0.1, 0.995 * r]) + 1.995 * r * cell + rng.uniform(-1e-3, 1e-3, (n, 3)) * r
    pos[:, 3] = r
    scene.pos[...] = pos.reshape(scene.pos.shape)
    scene.vel[...] = rng.uniform(-0.05, 0.05, (n, 3)).reshape(scene.vel.shape)
    return scene, rng


@pytest.mark.parametrize("n,capacity", [(1, 12), (7, 16), (8, 6), (9, 16), (17, 12), (33, 16)])
def test_gradient_at_the_edges_of_the_lane_groups(n, capacity):
    print(f"[calib lanes] n={n} capacity={capacity}", flush=True)
    scene, rng = lattice(n)
    w = rng.uniform(-1.0, 1.0, (n, 3))
    steps, h = 40, 1e-8
    cal = Calibration(scene, max_steps=steps, checkpoint_every=15, capacity=capacity)
    th = np.array([scene.cp_pp.fric, scene.cp_pp.rest, np.log(scene.cp_pp.Ei)])
    fd = np.zeros(3)
    for k in range(3):
        tp, tm = th.copy(), th.copy()
        tp[k] += h
        tm[k] -= h
        fd[k] = np.sum(w * (cal.forward(tp, steps)[:, :3] - cal.forward(tm, steps)[:, :3])) / (2 * h)
    cal.forward(th, steps)
    grad = cal.backward(w)
    print(f"[calib lanes] adjoint={grad} central differences={fd}", flush=True)
    assert np.abs(fd).max() > 0.0
    assert np.abs(grad - fd).max() <= 1e-3 * np.abs(fd).max(), (grad, fd)
    assert cal.error_word() == 0
    cal.close()


@pytest.mark.parametrize("n,side,cell,quirks", [(1, 4, 1.0, None), (3, 4, 1.0, dict(stale_ft=1)),
                                                (1025, 10, 0.8, dict(gpu_force_law=1)), (2100, 12, 1.0, None),
                                                (34001, 48, 1.0, None)])
def test_forward_is_the_oracle_for_every_wave_size_and_table(n, side, cell, quirks):
    print(f"[calib lanes] forward n={n} cell={cell} quirks={quirks}", flush=True)
    scene, _ = lattice(n, side)
    scene.cell_size *= cell
    steps = 8 if n < 10000 else 3
    cal = Calibration(scene, max_steps=steps, quirks=quirks)
    cal.forward(np.array([scene.cp_pp.fric, scene.cp_pp.rest, np.log(scene.cp_pp.Ei)]), steps)
    ref = xdem_ref.RefSim(scene, quirks=quirks)
    ref.step(steps)
    for name, g, r in zip(("pos", "vel", "ep", "ev"), cal.state(), (ref.pos, ref.vel, ref.ep, ref.ev)):
        assert np.array_equal(g, r), name
    assert ref.pp_count.max() > 2 if n > 10 else True
    assert cal.error_word() == 0
    cal.close()
