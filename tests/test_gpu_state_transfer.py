"""Node states in and out of a scene: bodies smaller and larger than a
workgroup's share and than the halves of the staging memory they pass
through, one of several bodies, positions or velocities alone, settings given
again between calls. Bar: the same doubles come back, and the scene steps
from them as one built with them does."""
import numpy as np
import pytest

import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def separate_tets(k):
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]]
    xyz = (p[None] + np.float32([0.3, 0.0, 0.0]) * np.arange(k, dtype=np.float32)[:, None, None]).reshape(-1, 3)
    return xyz.astype(np.float32).ravel(), np.arange(4 * k, dtype=np.uint32)


# 4 k nodes: around 256 (a workgroup), 43,690 (a half of the staging memory), and several halves
@pytest.mark.parametrize("k", [1, 63, 64, 65, 10922, 10923, 21846, 33000])
def test_round_trip(ctx, k):
    xyz, tets = separate_tets(k)
    sc = xf.Scene(ctx)
    first = xf.tet_block(2, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    sc.add_body(*first, 1000.0)
    b = sc.add_body(xyz, tets, 1000.0)
    sc.finalize()
    before = sc.get_state(0)
    r = np.random.RandomState(k)
    x, v = r.normal(size=xyz.size), r.normal(size=xyz.size)
    sc.set_state(b, x, v)
    xg, vg = sc.get_state(b)
    assert np.array_equal(xg, x) and np.array_equal(vg, v)
    x2, v2 = x + 1.0, v - 1.0
    sc.set_state(b, x=x2)
    assert np.array_equal(sc.get_state(b)[0], x2) and np.array_equal(sc.get_state(b)[1], v)
    sc.set_state(b, v=v2)
    only = np.zeros(xyz.size)
    ctx.check(xf.lib().xf_scene_get_state(sc.h, b, only.ctypes.data, None), "x only")
    assert np.array_equal(only, x2)
    ctx.check(xf.lib().xf_scene_get_state(sc.h, b, None, only.ctypes.data), "v only")
    assert np.array_equal(only, v2)
    ctx.check(xf.lib().xf_scene_get_state(sc.h, b, None, None), "neither")
    for a, c in zip(before, sc.get_state(0)):
        assert np.array_equal(a, c)
    sc.close()


def test_steps_from_a_set_state(ctx):
    """Positions, velocities, pins and inverse masses after set_state: the
    next frames equal those of a scene that starts there."""
    wl = workloads.beam_neo_12x4x4(energy=7)
    dt, S = float(wl["dt"]), wl["substeps"]
    a = workloads.make_scene(ctx, wl)
    a.step(S, dt)
    x, v = a.get_state(0)
    a.step(S, dt)
    b = workloads.make_scene(ctx, wl)
    b.set_state(0, x, v)
    b.set_time(a.time() / 2)
    b.step(S, dt)
    for p, q in zip(a.get_state(0), b.get_state(0)):
        assert np.array_equal(p, q)
    a.close()
    b.close()


def test_settings_given_again(ctx):
    """The same settings, settings that only touch the nodes, and settings
    that change the material, given between steps, act as in a scene that
    gets each for the first time."""
    wl = workloads.beam_neo_12x4x4(energy=4)
    dt = float(wl["dt"])
    sequence = [dict(), dict(), dict(gravity=(1.0, -5.0)), dict(gravity=(1.0, -5.0), compliance=4e-5),
                dict(gravity=(1.0, -5.0), compliance=4e-5), dict(damping=0.02, rayleigh_type=2), dict(),
                dict(poissons_ratio=0.4), dict(yeoh=(0.2, 0.1, 0.1), energy=7)]
    sc = workloads.make_scene(ctx, wl)
    x, v = sc.get_state(0)
    t = 0.0
    for change in sequence:
        sc.set_settings(0, **dict(wl["settings"], **change))
        sc.step(3, dt)
        fresh = workloads.make_scene(ctx, dict(wl, settings=dict(wl["settings"], **change)))
        fresh.set_state(0, x, v)
        fresh.set_time(t)
        fresh.step(3, dt)
        x, v = fresh.get_state(0)
        fresh.close()
        t = sc.time()
        for p, q in zip(sc.get_state(0), (x, v)):
            assert np.array_equal(p, q), change
    sc.close()
