"""The cohesive pair predicate at its edge: a separated pair attracts while its gap is below the JKR
separation depth 3/4 x^(1/3) (impl:415-423, 708-718). Pairs are laid at the gaps nearest the depth,
a few roundings of the distance either side; the depth is of the size of a radius, where a
rounding of the distance is one to four of the depth's. Every decision is that of the reference's
expression, 3/4 pow(x, 1.0 / 3.0) with the device's pow, and the exact one wherever the gap is
more than two units in the last place from the depth of the double x (one for the power's
error, a half for the product's, rounded up)."""
import ctypes as C
from decimal import Decimal, getcontext

import numpy as np
import pytest

from test_gpu_launchers import Arrays, call, dev, host, ptr, setup_params
import xdem_ref
from xdynamics_dll_amd import DemContext, SceneData, contact_property

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

E, NU, COH = 1.0e5, 0.3, 38.0


def gap_of(ri, rj, d):
    return -((ri + rj) - np.sqrt(d * d))


def edge_pairs(n, seed=3):
    """(ri, rj, d, x, gap, passes, sure) of n pairs of radii at 9 distances each."""
    getcontext().prec = 40
    rng = np.random.default_rng(seed)
    pi = 3.14159265358979323846
    eq = 1.0 / (((1.0 - NU * NU) / E) + ((1.0 - NU * NU) / E))
    pcc, ee = pi * pi * COH * COH, eq * eq
    out = []
    for _ in range(n):
        ri, rj = rng.uniform(0.8e-3, 1.2e-3, 2)
        x = (pcc * ((ri * rj) / (ri + rj))) / ee
        depth = Decimal(3) / 4 * Decimal(x) ** Decimal(1.0 / 3.0)
        f = float(depth)
        d0 = (ri + rj) + f
        ds = [d0]
        for way in (-np.inf, np.inf):
            d = d0
            for _ in range(3):
                d = np.nextafter(d, way)
                ds.append(d)
        ds += [(ri + rj) + f * (1.0 - 1e-6), (ri + rj) + f * (1.0 + 1e-9)]
        for d in ds:
            gap = Decimal(float(gap_of(ri, rj, d)))
            out.append((ri, rj, d, x, float(gap), gap < depth, abs(gap - depth) > 2 * Decimal(float(np.spacing(f)))))
    return [np.array(c) for c in zip(*out)]


def scene_of(ri, rj, d):
    """Pair k at (0, y_k, z_k) and (d, y_k, z_k), rows far apart."""
    m = len(d)
    k, side = np.arange(m), int(np.ceil(np.sqrt(m)))
    y, z = (k % side) * 0.009 - 0.5, (k // side) * 0.009 - 0.5
    pos = np.zeros((2 * m, 4))
    pos[0::2] = np.stack([np.zeros(m), y, z, ri], axis=1)
    pos[1::2] = np.stack([d, y, z, rj], axis=1)
    cp = contact_property(E, E, NU, NU, 0.5, 0.4, 0.02, COH)
    scene = SceneData.from_positions(pos, 2500.0, cp, walls=(), dt=1e-9, vel=np.zeros((2 * m, 3)), gravity=(0.0, 0.0, 0.0))
    scene.cell_size = 4.0e-3
    return scene


def check(count, passes, sure, rounded, what):
    hit = count[0::2] > 0
    print(f"[cohesion edge] {what}: {len(hit)} pairs, {int((hit != rounded).sum())} not the expression's, "
          f"{int((hit != passes)[sure].sum())} wrong off the edge, {int((hit != passes)[~sure].sum())} at it", flush=True)
    assert np.array_equal(count[0::2], count[1::2])
    assert not (hit != passes)[sure].any()
    assert np.array_equal(hit, rounded)
    assert passes.any() and not passes.all()


def test_predicate_at_the_separation_depth():
    ri, rj, d, x, gap, passes, sure = edge_pairs(600)
    rounded = gap < host((3.0 / 4.0) * torch.pow(dev(x), 1.0 / 3.0))
    scene = scene_of(ri, rj, d)
    ref = xdem_ref.RefSim(scene)
    a = Arrays(ref)
    setup_params(scene)
    n = scene.np
    cp = dev(np.frombuffer(bytes(scene.cp_pp), dtype=np.float64).copy())
    call("xdem_reserve_workspace", n)
    call("xdem_cu_calculateHashAndIndex", ptr(a.hash), ptr(a.index), ptr(a.pos), 0, n)
    call("xdem_cu_reorderDataAndFindCellStart", ptr(a.hash), ptr(a.index), ptr(a.cstart), ptr(a.cend), ptr(a.sorted), n, ref.ncell)
    call("xdem_cu_calculate_p2p", ptr(a.pos), ptr(a.ep), ptr(a.vel), ptr(a.ev), ptr(a.force), ptr(a.moment), ptr(a.mass),
         ptr(a.tmax), ptr(a.rres), ptr(a.pp_count), ptr(a.pp_id), ptr(a.pp_tsd), ptr(a.sorted), ptr(a.cstart), ptr(a.cend),
         ptr(cp), n)
    torch.cuda.synchronize()
    check(host(a.pp_count, np.uint32), passes, sure, rounded, "launcher")
    w = C.c_uint()
    call("xdem_get_error_word", C.byref(w), 1)
    assert w.value == 0
    for fuse in (False, True):
        ctx = DemContext(scene, precision="fp64", fuse_velocity=fuse)
        ctx.step(1)     # at rest without gravity: the first step's positions are the given ones
        assert np.array_equal(ctx.read("pos")[:, :3], scene.pos[:, :3]) or fuse
        check(ctx.history("p2p")[0], passes, sure, rounded, f"context, fuse={fuse}")
        assert ctx.error_word() == 0
        ctx.close()
