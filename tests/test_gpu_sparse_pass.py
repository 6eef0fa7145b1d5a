"""Steps whose candidates are none, few or many, over several list builds: k_touch divides its work
by the totals that the lite pass of the last build step left, tests a sphere in one lane or in a
group of lanes by the lists' lengths (up to 6 entries, 18 at the largest skin), and leaves waves without one to
test at once. FP64 states are the oracle's, bit for bit, and the pair and wall contacts as many."""
import numpy as np
import pytest

import xdem_ref
from xdynamics_dll_amd import DemContext, SceneData, box_walls, contact_property

pytestmark = pytest.mark.gpu


def falling(n, touching, pitch, seed=5, speed=2.0):
    """n spheres a pitch apart falling on a floor, of which the first `touching` rows of the lattice
    overlap the floor or each other from the start; the speed brings more to it step by step."""
    rng = np.random.default_rng(seed)
    side = max(1, int(np.ceil(n ** (1.0 / 3.0))))
    k, rest = np.divmod(np.arange(n), side * side)
    j, i = np.divmod(rest, side)
    r = 1.0e-3
    p = np.stack([i * pitch + 2e-3, j * pitch + 2e-3, k * pitch + (0.999e-3 if touching else 1.004e-3)], axis=1)
    p[:, :2] += rng.uniform(-2e-6, 2e-6, (n, 2))
    pos = np.concatenate([p, np.full((n, 1), r)], axis=1)[rng.permutation(n)]
    vel = np.tile([0.0, 0.0, -speed], (n, 1)) + rng.uniform(-0.05, 0.05, (n, 3))
    L = side * pitch + 4e-3
    return SceneData.from_positions(pos, 2500.0, contact_property(1e7, 1e7, 0.3, 0.3, 0.3, 0.3, 0.01), walls=box_walls(L, L, 2 * L),
                                    dt=1e-6, vel=vel)


@pytest.mark.parametrize("fuse,skin", [(True, 0.0), (False, 0.0), (True, 2.0e-5), (False, 1.0e-3), (True, 1.0e-3)])
@pytest.mark.parametrize("n,touching,pitch", [(1, False, 2.1e-3), (63, False, 2.004e-3), (500, True, 2.4e-3),
                                              (4097, False, 2.002e-3), (4097, True, 1.998e-3), (20001, False, 2.3e-3)])
def test_candidates_come_and_go(n, touching, pitch, fuse, skin):
    print(f"[sparse pass] n={n} touching={touching} pitch={pitch} fuse={fuse} skin={skin}", flush=True)
    scene = falling(n, touching, pitch)
    gpu = DemContext(scene, precision="fp64", fuse_velocity=fuse, skin=skin, p2p_capacity=32)
    ref = xdem_ref.RefSim(scene)
    full = []
    for target in (1, 6, 14, 24) if n < 10000 else (2, 12):
        steps = target - gpu.info()["steps_done"]
        gpu.step(steps)
        ref.step(steps)
        for f in ("pos", "vel", "acc", "ep", "ev", "ea"):
            assert np.array_equal(gpu.read(f), getattr(ref, f)), (target, f)
        assert gpu.contact_count() == (int(ref.pp_count.sum()), int(ref.pl_count.sum()))
        full.append(gpu.info()["contact_spheres"])
    info = gpu.info()
    print(f"[sparse pass] full passes {full}, builds {info['list_builds']}, candidates {info['list_spheres']}", flush=True)
    assert gpu.error_word() == 0
    gpu.close()
