"""A mesh whose proxy spheres are larger than the spheres enlarges the reference's cell
(xDiscreteElementMethodSimulation.cpp:91-100), which fixes the order of the sphere contacts, also of
spheres that never meet the mesh: FP64 states and pair slots, in their order, are the oracle's, bit
for bit, with cells of 1, 2 and 9 times the spheres' own."""
import numpy as np
import pytest

import xdem_ref
from scenes import compressed_lattice, random_pack
from xdynamics_dll_amd import DemContext, contact_property

pytestmark = pytest.mark.gpu


def far_mesh(scene, size):
    """Two triangles of the given size, 0.2 m above the spheres, on a resting body."""
    t = np.array([[[0, 0, 0], [size, 0, 0], [size, size, 0]], [[0, 0, 0], [size, size, 0], [0, size, 0]]], dtype=np.float64)
    dbi = np.zeros(15)
    dbi[0], dbi[7] = 10.0, 1.0
    dbi[1:4] = (0.0, 0.0, scene.pos[:, 2].max() + 0.2)
    return t, dbi, contact_property(1e9, 5e7, 0.3, 0.25, 0.4, 0.6, 0.05)


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("make,size", [(compressed_lattice, 1e-3), (compressed_lattice, 6e-3), (random_pack, 8e-3), (random_pack, 4e-2)])
def test_order_of_the_contacts_under_an_enlarged_cell(make, size, fuse):
    scene = make()
    tris, dbi, cp = far_mesh(scene, size)
    ref = xdem_ref.RefSim(scene)
    ref.add_mesh(tris, dbi, cp)
    print(f"[mesh cell] {make.__name__} np={scene.np} fuse={fuse} cell {scene.cell_size:g} -> {ref.prm.cell_size:g}", flush=True)
    gpu = DemContext(scene, precision="fp64", fuse_velocity=fuse, meshes=[(0, tris, dbi, cp)])
    for steps in (1, 3, 20):
        gpu.step(steps)
        ref.step(steps)
        count, ids, tsd = gpu.history("p2p")
        assert np.array_equal(count, ref.pp_count)
        used = np.arange(ids.shape[1])[None, :] < count[:, None]
        assert np.array_equal(ids[used], ref.pp_id[:, : ids.shape[1]][used])
        for f in ("pos", "vel", "acc", "ep", "ev", "ea"):
            assert np.array_equal(gpu.read(f), getattr(ref, f)), (steps, f)
    assert count.sum() > scene.np // 4
    assert gpu.error_word() == 0
    gpu.close()
