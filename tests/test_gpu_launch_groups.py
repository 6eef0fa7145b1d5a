"""The launcher layer at the sizes where its division of work changes: the sphere launcher in
groups of 2 to 16 particles a wave (more candidates and contacts than a round, a half or the slots
hold). Integers are exact; sums and slots agree to 1e-12 of the largest (the material
constants come from the device's log and the host's: a rounding of a term, at most 18 terms a sum)."""
import ctypes as C

import numpy as np
import pytest

import xdem_ref
from test_gpu_launchers import Arrays, call, dev, host, ptr, setup_params
from xdynamics_dll_amd import _lib, SceneData, box_walls, contact_property

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("coh", [0.0, 0.05])
@pytest.mark.parametrize("n, pitch", [(1, 1.98e-3), (2, 1.98e-3), (27, 1.2e-3), (2049, 1.98e-3), (4099, 1.55e-3),
                                      (40001, 1.99e-3)])
def test_sphere_launcher(n, pitch, coh):
    """At a pitch of 1.2 mm second neighbours overlap too: up to 18 contacts a sphere, past the 12
    slots, and over 64 pairs a group; at 1.55 mm six deep ones."""
    rng = np.random.default_rng(n)
    side = max(1, int(np.ceil(n ** (1.0 / 3.0))))
    k, rest = np.divmod(np.arange(n), side * side)
    j, i = np.divmod(rest, side)
    p = np.stack([i, j, k], axis=1) * pitch + 3e-3 + rng.uniform(-2e-6, 2e-6, (n, 3))
    pos = np.concatenate([p, np.full((n, 1), 1.0e-3)], axis=1)[rng.permutation(n)]
    L = side * pitch + 6e-3
    scene = SceneData.from_positions(pos, 2500.0, contact_property(1e7, 1e7, 0.3, 0.3, 0.5, 0.4, 0.02, coh),
                                     walls=box_walls(L, L, L), dt=1e-6, vel=rng.normal(0.0, 0.05, (n, 3)))
    ref = xdem_ref.RefSim(scene)
    d = Arrays(ref)
    setup_params(scene)
    cp = dev(np.frombuffer(bytes(scene.cp_pp), dtype=np.float64).copy())
    for _ in range(2):    # the second launch reads the slots of the first
        call("xdem_cu_calculateHashAndIndex", ptr(d.hash), ptr(d.index), ptr(d.pos), 0, n)
        call("xdem_cu_reorderDataAndFindCellStart", ptr(d.hash), ptr(d.index), ptr(d.cstart), ptr(d.cend), ptr(d.sorted),
             n, ref.ncell)
        call("xdem_cu_calculate_p2p", ptr(d.pos), ptr(d.ep), ptr(d.vel), ptr(d.ev), ptr(d.force), ptr(d.moment),
             ptr(d.mass), ptr(d.tmax), ptr(d.rres), ptr(d.pp_count), ptr(d.pp_id), ptr(d.pp_tsd), ptr(d.sorted),
             ptr(d.cstart), ptr(d.cend), ptr(cp), n)
        ref.grid()
        over = xdem_ref.lib().ref_calculate_p2p(*p2p_args(ref))
        torch.cuda.synchronize()
        for name in ("force", "moment", "tmax", "rres"):
            close(host(getattr(d, name)), getattr(ref, name), name)
        count = host(d.pp_count, np.uint32)
        assert np.array_equal(count, ref.pp_count)
        used = np.arange(12)[None, :] < count[:, None]
        assert np.array_equal(host(d.pp_id, np.uint32)[used], ref.pp_id[used])
        close(host(d.pp_tsd)[used], ref.pp_tsd[used], "slots")
    word = C.c_uint()
    call("xdem_get_error_word", C.byref(word), 1)
    assert word.value == (_lib.ERR_P2P_OVERFLOW if over else 0), hex(word.value)
    assert bool(over) == (pitch == 1.2e-3)


def close(a, b, name):
    a, b = np.asarray(a).reshape(-1), np.asarray(b).reshape(-1)
    if b.size:
        assert np.abs(a - b).max() <= 1e-12 * max(np.abs(b).max(), 1e-300), name


def p2p_args(ref):
    P = xdem_ref._p
    return (C.byref(ref.prm), C.byref(ref.q), P(ref.pos), P(ref.ep), P(ref.vel), P(ref.ev), P(ref.force), P(ref.moment),
            P(ref.mass), P(ref.tmax), P(ref.rres), P(ref.pp_count), P(ref.pp_id), P(ref.pp_tsd), P(ref.sorted_index),
            P(ref.cstart), P(ref.cend), C.byref(ref.cp_pp), ref.np, 12)
