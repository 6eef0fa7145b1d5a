"""Scenes of which a part is touched: the pair-test and contact kernels take their spheres by sweeping
the sorted slots from half of them on, in scenes of 65,536 spheres or more from three quarters, and
else from a queue, at least 4 to 32 spheres to a wave by how many are untouched. FP64 states,
histories and counts are the oracle's at both sides of each line. A step's time grows as the touched
spheres do: of 1,000,000 with 55 percent touched at most 1.22 (55 / 45) times that with 45 percent,
and a fifth more for what else differs."""
import time

import numpy as np
import pytest

import xdem_ref
from test_gpu_full_pass import pack
from xdynamics_dll_amd import DemContext, SceneData, box_walls, contact_property

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("n,part", [(400, 0.49), (400, 0.51), (9001, 0.3), (65535, 0.51), (65536, 0.55), (65537, 0.74),
                                    (66001, 0.76), (70001, 0.38), (70001, 0.42)])
def test_partly_touched_scene_is_the_oracle(n, part, fuse):
    touching = int(n * part)
    scene = pack(touching, n - touching)
    print(f"[partly touched] {touching} of {n}, fuse={fuse}", flush=True)
    ref = xdem_ref.RefSim(scene)
    ref.step(3)
    # full_blocks 64: few waves of many spheres, several rounds
    for blocks in (0, 64):
        gpu = DemContext(scene, precision="fp64", fuse_velocity=fuse, p2p_capacity=12, full_blocks=blocks)
        gpu.step(3)
        for f in ("pos", "vel", "acc", "ep", "ev", "ea"):
            assert np.array_equal(gpu.read(f), getattr(ref, f)), (blocks, f)
        count, ids, _ = gpu.history("p2p")
        assert np.array_equal(count, ref.pp_count)
        used = np.arange(ids.shape[1])[None, :] < count[:, None]
        assert np.array_equal(ids[used], ref.pp_id[:, : ids.shape[1]][used])
        assert gpu.contact_count() == (int(ref.pp_count.sum()), int(ref.pl_count.sum()))
        assert gpu.error_word() == 0
        gpu.close()


def layered(n, touching, pitch=3.0e-3):
    """A compressed lattice of `touching` spheres on the floor and the other spheres above it, free."""
    rng = np.random.default_rng(7)
    side, wide = (max(1, int(np.ceil(m ** (1.0 / 3.0)))) for m in (touching, n - touching))

    def lattice(m, s):
        k, rest = np.divmod(np.arange(m), s * s)
        j, i = np.divmod(rest, s)
        return np.stack([i, j, k], axis=1)

    p = lattice(touching, side) * 1.985e-3 + np.array([1.2e-3, 1.2e-3, 1.0e-3 - 1e-6]) + rng.uniform(-5e-6, 5e-6, (touching, 3))
    q = lattice(n - touching, wide) * pitch + np.array([3e-3, 3e-3, p[:, 2].max() + 10e-3])
    pos = np.concatenate([np.concatenate([p, q]), np.full((n, 1), 1.0e-3)], axis=1)[rng.permutation(n)]
    L = max(side * 2.0e-3, wide * pitch) + 4e-3
    return SceneData.from_positions(pos, 2500.0, contact_property(1e7, 1e7, 0.3, 0.3, 0.3, 0.3, 0.01),
                                    walls=box_walls(L, L, pos[:, 2].max() + 10e-3), dt=1e-6, vel=rng.uniform(-0.05, 0.05, (n, 3)))


def test_time_grows_as_the_touched_spheres():
    n, us = 1000000, []
    for part in (0.45, 0.55):
        gpu = DemContext(layered(n, int(n * part)), precision="mixed", p2p_capacity=16, fuse_velocity=True, step_graph=20)
        times = []
        for _ in range(6):
            gpu.synchronize()
            t = time.perf_counter()
            gpu.step(20)
            gpu.synchronize()
            times.append((time.perf_counter() - t) / 20 * 1e6)
        assert gpu.error_word() == 0
        us.append(min(times[2:]))
        gpu.close()
    print(f"[partly touched] us a step {us}", flush=True)
    assert us[1] <= 1.22 * 1.2 * us[0]
