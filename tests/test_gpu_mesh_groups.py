"""The triangle launcher at the sizes where its division of work changes: 4 and 16 particles to a
wave, a last group that is not full, and more than 20 candidates of one kind at a sphere (a terrain
of 0.1 mm triangles; the lists of 20 fill, as the reference's). Counts and ids are the oracle's;
sums and slots agree to 1e-12 of the largest (the material constants come from the device's log and
the host's: a rounding of a term, at most 20 terms a sum)."""
import ctypes as C

import numpy as np
import pytest

import xdem_ref
from mesh_scenes import body_pose, fit_proxies, mesh_scene, terrain, triangle_infos
from test_gpu_launchers import call, dev, host, ptr
from xdynamics_dll_amd import SceneData, _lib, contact_property

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
CAP, NCELL = 5, 128 ** 3


def many(n, coh):
    """n spheres at the places of a scene of 397, each with a shift of up to 10 nm."""
    base, tris, prox, dbi, cp = mesh_scene(n=397, coh=coh)
    rng = np.random.default_rng(n)
    pick = rng.integers(0, base.np, n)
    pos = base.pos[pick].copy()
    pos[:, :3] += rng.uniform(-1e-8, 1e-8, (n, 3))
    scene = SceneData.from_positions(pos, 2500.0, cp, walls=(), dt=1e-5, vel=base.vel[pick])
    scene.cell_size = base.cell_size
    return scene, tris, prox, dbi, cp


def fine(n):
    """Spheres overlapping a nearly flat terrain of 0.1 mm triangles by up to a tenth of a radius."""
    rng = np.random.default_rng(n)
    h, nx = 1.0e-4, 40
    tris = terrain(nx=nx, h=h, amp=2e-8)
    dbi = body_pose()
    dbi[1:4], dbi[7:11], dbi[11:15] = 0.0, (1.0, 0.0, 0.0, 0.0), 0.0
    r = rng.uniform(0.8e-3, 1.2e-3, n)
    xy = rng.uniform(1.2e-3, nx * h - 1.2e-3, (n, 2))
    pos = np.column_stack([xy, r * rng.uniform(0.9, 0.999, n), r])
    cp = contact_property(4e7, 2e8, 0.28, 0.3, 0.45, 0.55, 0.03, 0.0)
    scene = SceneData.from_positions(pos, 2500.0, cp, walls=(), dt=1e-5, vel=rng.normal(0, 0.03, (n, 3)))
    return scene, tris, fit_proxies(tris), dbi, cp


@pytest.mark.parametrize("make,n,coh,full", [(many, 4099, 0.0, False), (many, 4099, 0.05, False), (many, 30011, 0.0, False),
                                             (fine, 7, 0.0, True), (fine, 5000, 0.0, True)])
def test_mesh_launcher(make, n, coh, full):
    scene, tris, prox, dbi, cp = make(n, coh) if make is many else make(n)
    nt = len(tris)
    print(f"[mesh groups] {make.__name__} n={n} ntri={nt} coh={coh}", flush=True)
    L, prm, q = xdem_ref.lib(), scene.dem_parameters(), xdem_ref.quirks_struct({})
    rng = np.random.default_rng(1)
    ep = np.zeros((n, 4))
    ep[:, 0] = 1.0
    ev = rng.normal(size=(n, 4)) * 0.5
    ev[:, 0] = 0.0
    cnt, ids, tsd = np.zeros(n, np.uint32), np.zeros((n, CAP), np.uint32), np.zeros((n, CAP, 2))
    cnt[::3] = 2     # a step's history before
    ids[::3, :2] = rng.integers(0, nt, (len(cnt[::3]), 2))
    tsd[::3, :2] = rng.normal(size=(len(cnt[::3]), 2, 2)) * 1e-6
    vlist, local = np.ascontiguousarray(tris.reshape(nt, 9)), np.ascontiguousarray(prox[:, :3])
    sph = np.zeros((nt, 4))
    sph[:, 3] = prox[:, 3]
    g = {k: dev(v) for k, v in dict(vlist=vlist, local=local, sph=sph, dbi=dbi, pos=scene.pos, ep=ep, vel=scene.vel, ev=ev,
                                    force=np.zeros((n, 3)), moment=np.zeros((n, 3)), mass=scene.mass, tmax=np.zeros((n, 3)),
                                    rres=np.zeros(n), cnt=cnt, ids=ids, tsd=tsd, hash=np.zeros(n + nt, np.uint32),
                                    index=np.zeros(n + nt, np.uint32), sorted=np.zeros(n + nt, np.uint32),
                                    cs=np.zeros(NCELL, np.uint32), ce=np.zeros(NCELL, np.uint32),
                                    cp=np.frombuffer(bytes(cp), dtype=np.float64).copy()).items()}
    g["tri"] = dev(np.frombuffer(bytes(triangle_infos(nt)), dtype=np.uint8).copy())
    bf = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(6)]
    p = {k: ptr(v) for k, v in g.items()}
    prm.nsphere = nt
    word = C.c_uint()
    call("xdem_setDEMSymbolicParameter", C.byref(prm))
    call("xdem_set_quirks", C.byref(_lib.Quirks(0, 0, 1, 1)))
    call("xdem_reserve_workspace", n + nt)
    call("xdem_get_error_word", C.byref(word), 1)
    call("xdem_cu_update_meshObjectData", p["vlist"], p["sph"], p["local"], p["tri"], p["dbi"], nt)
    call("xdem_cu_calculateHashAndIndex", p["hash"], p["index"], p["pos"], 0, n)
    call("xdem_cu_calculateHashAndIndexForPolygonSphere", p["hash"], p["index"], n, nt, p["sph"])
    call("xdem_cu_reorderDataAndFindCellStart", p["hash"], p["index"], p["cs"], p["ce"], p["sorted"], n + nt, NCELL)
    call("xdem_set_body_force_buffers", *(ptr(b) for b in bf))
    call("xdem_cu_particle_polygonObject_collision", p["tri"], p["dbi"], p["pos"], p["ep"], p["vel"], p["ev"], p["force"],
         p["moment"], p["mass"], p["tmax"], p["rres"], p["cnt"], p["ids"], p["tsd"], p["sph"], p["sorted"], p["cs"], p["ce"],
         p["cp"], n, nt)
    torch.cuda.synchronize()
    call("xdem_get_error_word", C.byref(word), 1)
    # the oracle on the launcher's own cell table
    P = xdem_ref._p
    srt, cs, ce = (host(g[k], np.uint32).copy() for k in ("sorted", "cs", "ce"))
    tri = triangle_infos(nt)
    L.ref_update_mesh_object_data(P(dbi), P(vlist), P(sph), P(local), C.addressof(tri), nt)
    out = {k: np.zeros((n, 3)) for k in ("force", "moment", "tmax")}
    out["rres"], rbf, pos, vel, mass = np.zeros(n), [np.zeros(n) for _ in range(6)], scene.pos, scene.vel, scene.mass
    over = L.ref_particle_polygon_collision(C.byref(prm), C.byref(q), C.addressof(tri), P(dbi), *(P(b) for b in rbf), P(pos),
                                            P(ep), P(vel), P(ev), P(out["force"]), P(out["moment"]), P(mass), P(out["tmax"]),
                                            P(out["rres"]), P(cnt), P(ids), P(tsd), P(srt), P(cs), P(ce), C.byref(cp), n, nt, CAP)
    print(f"[mesh groups] contacts {int(cnt.sum())}, overflows {over}, error word {word.value:#x}", flush=True)
    assert cnt.sum() > n // 2
    assert np.array_equal(host(g["cnt"], np.uint32), cnt)
    used = np.arange(CAP)[None, :] < cnt[:, None]
    assert np.array_equal(host(g["ids"], np.uint32)[used], ids[used])
    for name, a, b in [("slots", host(g["tsd"])[used], tsd[used])] + [(k, host(g[k]), v) for k, v in out.items()] + \
            [(f"body {c}", host(bf[c]), rbf[c]) for c in range(6)]:
        assert np.abs(a - b).max() <= 1e-12 * max(np.abs(b).max(), 1e-300), name
    want = (_lib.ERR_MESH_LIST if full else 0) | (_lib.ERR_MESH_OVERFLOW if over else 0)
    assert word.value == want, hex(word.value)
