"""The full contact pass at the sizes where its division of work changes: a wave takes 1 to 64
touched spheres, by whether SIMDs get one wave or two, found by sweeping the sorted slots when half
of them (three quarters in large scenes) are touched; otherwise at least 4 to 32 from the queue. FP64 states and histories
are those of the oracle, bit for bit: the pass adds a sphere's pairs in the reference's order
whatever the division."""
import numpy as np
import pytest

import xdem_ref
from xdynamics_dll_amd import DemContext, SceneData, box_walls, contact_property

pytestmark = pytest.mark.gpu


def pack(n, free, seed=11):
    """n spheres: a compressed lattice on the floor of a box and, above it, `free` spheres more
    than a diameter apart that touch nothing."""
    rng = np.random.default_rng(seed)
    side = max(1, int(np.ceil(n ** (1.0 / 3.0))))
    k, rest = np.divmod(np.arange(n), side * side)
    j, i = np.divmod(rest, side)
    p = np.stack([i, j, k], axis=1) * 1.985e-3 + np.array([1.2e-3, 1.2e-3, 1.0e-3 - 1e-6])
    p += rng.uniform(-5e-6, 5e-6, p.shape)
    wide = max(1, int(np.ceil(free ** 0.5)))
    a, b = np.divmod(np.arange(free), wide)
    top = p[:, 2].max() + 10e-3
    q = np.stack([a * 6e-3 + 3e-3, b * 6e-3 + 3e-3, np.full(free, top)], axis=1)
    x = np.concatenate([p, q])
    pos = np.concatenate([x, np.full((len(x), 1), 1.0e-3)], axis=1)[rng.permutation(len(x))]
    cp = contact_property(1e7, 1e7, 0.3, 0.3, 0.3, 0.3, 0.01)
    L = max(side * 2.0e-3, wide * 6e-3) + 4e-3
    return SceneData.from_positions(pos, 2500.0, cp, walls=box_walls(L, L, top + 10e-3), dt=1e-6,
                                    vel=rng.uniform(-0.05, 0.05, (len(pos), 3)))


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("n, free", [(1, 0), (3, 4), (4, 0), (65, 200), (255, 0), (2049, 3000), (4097, 0),
                                     (9000, 12000), (31, 3000), (2113, 40000), (26011, 0), (70001, 0)])
def test_full_pass_equals_oracle(n, free, fuse):
    scene = pack(n, free)
    print(f"[full pass] {n} touching, {free} free, fuse={fuse}", flush=True)
    ref = xdem_ref.RefSim(scene)
    steps = 2 if n > 10000 else 5
    ref.step(steps)
    # 0: waves of as few spheres as fill the device; 1: always 64 spheres to a wave
    for merge in (0, 1):
        gpu = DemContext(scene, precision="fp64", fuse_velocity=fuse, p2p_capacity=12, merge_pairs_below=merge)
        gpu.step(steps)
        for f in ("pos", "vel", "acc", "ep", "ev", "ea"):
            assert np.array_equal(gpu.read(f), getattr(ref, f)), (merge, f)
        count, ids, tsd = gpu.history("p2p")
        assert np.array_equal(count, ref.pp_count)
        used = np.arange(ids.shape[1])[None, :] < count[:, None]
        assert np.array_equal(ids[used], ref.pp_id[:, : ids.shape[1]][used])
        assert np.array_equal(tsd[used], np.asarray(ref.pp_tsd).reshape(len(count), -1, 2)[:, : ids.shape[1]][used])
        n_pp, n_wall = gpu.contact_count()
        assert n_pp == int(ref.pp_count.sum()) and n_wall == int(ref.pl_count.sum())
        assert gpu.error_word() == 0
        gpu.close()
