"""Lanes per vertex ring left to the library (128, 64 or 32 by the rings of a
colour) and rings with more nodes and tets than are stored by the ring's
index. Bar: bit-exact with the oracle's serial ring sweep and with explicit
lanes per ring."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu

DAMPING = [dict(), dict(damping=0.02, rayleigh_type=0), dict(damping=0.02, rayleigh_type=1),
           dict(damping=0.02, rayleigh_type=2, pbd_damping=0.003), dict(damping=0.02, rayleigh_type=3)]


def workload(xyz, tets, energy, **settings):
    return dict(name="rings", xyz=xyz, tets=tets, density=1000.0,
                pinned=(np.asarray(xyz[0::3]) < np.asarray(xyz[0::3]).min() + 0.05).astype(np.uint8), velocity=None,
                tet_mu=None, settings=dict(dict(energy=energy, compliance=1e-6 if energy == 8 else 2e-5,
                                                poissons_ratio=0.45, gravity=(0.0, -9.81),
                                                collide=xf.COLLIDE_GROUND, ground_y=-0.35, friction=0.5), **settings),
                dt=np.float32(1.0) / np.float32(1200.0), substeps=4)


def fan(n):
    """A vertex in the middle of n points on a sphere, a tet to every face of
    their hull: a ring of n + 1 nodes and 2 n - 4 tets."""
    from scipy.spatial import ConvexHull
    k = np.arange(n) + 0.5
    z, phi = 1.0 - 2.0 * k / n, np.pi * (1.0 + 5.0 ** 0.5) * k
    p = np.stack([np.sqrt(1 - z * z) * np.cos(phi), np.sqrt(1 - z * z) * np.sin(phi), z], 1) * 0.3
    faces = ConvexHull(p).simplices
    x = np.concatenate([[[0.0, 0.0, 0.0]], p]).astype(np.float32)
    t = np.concatenate([np.zeros((len(faces), 1), int), faces + 1], 1)
    m = x[t]
    vol = np.linalg.det(m[:, 1:] - m[:, :1])
    cube, ct = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    c = np.asarray(cube).reshape(-1, 3)[np.asarray(ct).reshape(-1, 4)]
    want = np.sign(np.linalg.det(c[:, 1:] - c[:, :1]))[0]
    t[vol * want < 0] = t[vol * want < 0][:, [0, 2, 1, 3]]
    return x.ravel(), t.astype(np.uint32).ravel()


def run(ctx, wl, **opts):
    sc = workloads.make_scene(ctx, wl, **opts)
    for _ in range(2):
        sc.step(wl["substeps"], float(wl["dt"]))
    out = sc.get_state(0) + (sc.order(0)[0], sc.ring_order(0)[0])
    sc.close()
    return out


# 17: 30 tets, all by the index; 18: 32; 19: 34; 31, 32: as many nodes; 40: 76
# tets, more than the 64 lanes that take them in the widest team
@pytest.mark.parametrize("n", [4, 17, 18, 19, 31, 32, 40])
@pytest.mark.parametrize("damping", range(len(DAMPING)))
@pytest.mark.parametrize("energy", [8, 9, 10])
def test_large_rings_equal_oracle(ctx, n, damping, energy):
    wl = workload(*fan(n), energy, **DAMPING[damping])
    x, v, order, rorder = run(ctx, wl)
    ob = po.body_from_workload(wl, "ref64")
    ob.substep(po.params_from_settings(wl["dt"], wl["settings"]), order, count=2 * wl["substeps"], ring_order=rorder)
    assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V)
    for lanes in (16, 32):
        y = run(ctx, wl, ring_lanes=lanes)
        assert np.array_equal(x, y[0]) and np.array_equal(v, y[1])


# about 70, 700 and 2,000 rings a colour
@pytest.mark.parametrize("cells", [(10, 9, 11), (60, 15, 15), (80, 25, 22)])
@pytest.mark.parametrize("damping", [0, 1, 3])
def test_automatic_lanes_equal_explicit(ctx, cells, damping):
    xyz, tets = xf.tet_block(*cells, (0.1, 0.1, 0.1), (0.0, -0.2, -0.2))
    wl = workload(xyz, tets, 10, **DAMPING[damping])
    a = run(ctx, wl)
    for lanes in (16, 32):
        b = run(ctx, wl, ring_lanes=lanes)
        assert all(np.array_equal(p, q) for p, q in zip(a, b))
