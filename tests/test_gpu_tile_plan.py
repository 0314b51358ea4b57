"""When the tables of the tile launches are made: by the first step call that
could use them, never for a scene whose settings keep it on other routes, and
never by the allocation-free adjoint."""
import numpy as np
import pytest

import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def block(**settings):
    """A block that runs as tiles (3,900 nodes: no whole calls)."""
    wl = workloads.beam_yeoh(24, 12, 11, structured=False)
    return dict(wl, settings=dict(wl["settings"], collide=xf.COLLIDE_GROUND, **settings))


def held(sc):
    return sc.info()["device_bytes"]


@pytest.mark.parametrize("settings", [dict(energy=xf.ENERGY_CONTINUOUS_SKIN, poissons_ratio=0.45),
                                      dict(energy=xf.ENERGY_PIXAR), dict(energy=xf.ENERGY_CUBE_NEO),
                                      dict(volume_passes=1), dict(damping=0.02, rayleigh_type=2),
                                      dict(damping=0.02, rayleigh_type=0), dict(pbd_damping=0.002)])
def test_none_for_scenes_on_other_routes(ctx, settings):
    wl = block(**settings)
    plain = workloads.make_scene(ctx, wl, launch_mode=xf.LAUNCH_PERSISTENT)
    base = held(plain)
    plain.close()
    grown = []
    for forced in (False, True):
        sc = workloads.make_scene(ctx, wl)
        assert held(sc) == base
        sc.set_colour_launches(forced)
        for _ in range(2):
            sc.step(2, float(wl["dt"]))
        assert sc.route()[0] in (xf.ROUTE_COLOURS, xf.ROUTE_RINGS)
        grown.append(held(sc))
        sc.close()
    assert grown[0] == grown[1]


def test_made_by_the_first_call_that_uses_them(ctx):
    """Not while passes keep the scene off the route; once, then."""
    wl = block()
    dt = float(wl["dt"])
    sc = workloads.make_scene(ctx, wl)
    sc.set_settings(0, **dict(wl["settings"], damping=0.02, rayleigh_type=2))
    sc.step(2, dt)
    before = held(sc)
    sc.set_settings(0, **wl["settings"])
    sc.step(2, dt)
    assert sc.route()[0] == xf.ROUTE_TILES and held(sc) > before
    after = held(sc)
    sc.step(3, dt)
    sc.profile(1, dt)
    assert sc.route()[0] == xf.ROUTE_TILES and held(sc) == after
    sc.close()


@pytest.mark.parametrize("slots", ["none", "before", "after"])
def test_allocation_free_adjoint_makes_none(ctx, slots):
    """The allocation-free adjoint neither plans nor allocates, with the
    material slots made before the plan, after it, or not at all, and gives
    what the other entry point gives."""
    wl = block()
    dt = float(wl["dt"])
    at = np.array([4, 8], np.uint32)
    x0 = np.asarray(wl["xyz"], np.float64)
    tg = np.tile(x0, (2, 1))
    tg[:, 1::3] -= 0.01
    got = []
    for noalloc in (True, False):
        sc = workloads.make_scene(ctx, wl)
        L0 = sc.adjoint(8, dt, at, tg, window=4, noalloc=noalloc)
        assert sc.route()[0] == (xf.ROUTE_COLOURS if noalloc else xf.ROUTE_TILES)
        if slots == "before":
            sc.set_settings(0, **dict(wl["settings"], volume_passes=1))
            sc.step(1, dt)
        sc.set_settings(0, **wl["settings"])
        sc.step(1, dt)
        assert sc.route()[0] == xf.ROUTE_TILES
        if slots == "after":
            sc.set_settings(0, **dict(wl["settings"], volume_passes=1))
            sc.step(1, dt)
        if slots != "none":
            sc.set_settings(0, **dict(wl["settings"], poissons_ratio=0.47))
        sc.set_state(0, x0, np.zeros(x0.size))
        size = held(sc)
        L1 = sc.adjoint(8, dt, at, tg, window=4, noalloc=noalloc)
        assert sc.route()[0] == xf.ROUTE_TILES
        if noalloc:
            assert held(sc) == size
        got.append(L0 + L1 + sc.get_state(0))
        sc.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_autotuned_block_scene_keeps_none(ctx):
    """Tuning times the per-colour mode too; its tables go with it unless it
    is the choice, and are then used."""
    wl = block()
    sc = workloads.make_scene(ctx, wl, sweep_blocks=True, launch_mode=xf.LAUNCH_BLOCKS)
    mode, _, _ = sc.autotune(3, float(wl["dt"]), reps=1)
    first = held(sc)
    sc.step(2, float(wl["dt"]))
    if mode == xf.LAUNCH_PER_COLOUR:
        assert sc.route()[0] in (xf.ROUTE_TILES, xf.ROUTE_COLOURS)
    else:
        plain = workloads.make_scene(ctx, wl, sweep_blocks=True, launch_mode=xf.LAUNCH_BLOCKS,
                                     block_lanes=sc.info()["block_lanes"])
        # within the slot tables, which the tuner repacks (a tile entry is 76 bytes)
        assert abs(first - held(plain)) < 76 * 4 * 24 * 12 * 11
        plain.close()
    sc.close()
