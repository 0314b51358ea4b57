"""One launch per colour where the library would take another route
(xf_scene_set_colour_launches), and the route that a step call took
(xf_scene_get_route). The kernels of a launch per colour still run large
scenes, large damped bodies and held nodes; here they run small ones, bit for
bit against the oracle's serial sweep in the reported order."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def forced(ctx, wl, **opts):
    sc = workloads.make_scene(ctx, wl, **opts)
    sc.set_colour_launches()
    return sc


def check(sc, wl, calls, block, tick=0):
    """The scene after step calls of `calls` substeps equals the oracle, by
    launches per colour of `block` threads."""
    sc.set_tick(tick)
    for n in calls:
        sc.step(n, float(wl["dt"]))
    assert sc.route() == (xf.ROUTE_COLOURS, block)
    x, v = sc.get_state(0)
    ob = po.body_from_workload(wl, "ref64")
    ob.tick = tick
    ob.substep(po.params_from_settings(wl["dt"], wl["settings"]), sc.order(0)[0], count=sum(calls))
    assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V)


@pytest.mark.parametrize("block", [64, 128, 192, 256])
@pytest.mark.parametrize("energy,sim", [(3, True), (4, True), (5, True), (6, True), (7, True), (4, False),
                                        (5, False), (7, False)])
def test_workgroup_sizes(ctx, energy, sim, block):
    wl = workloads.beam_neo_12x4x4(energy=energy, simultaneous=sim)
    sc = forced(ctx, wl, block_size=block)
    check(sc, wl, (7, 2), block)
    sc.close()


@pytest.mark.parametrize("energy,sim", [(4, True), (7, True), (4, False), (3, True)])
@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("passes", [0, 1, 2])
def test_slabs_and_volume_passes(ctx, energy, sim, block, passes):
    wl = workloads.beam_neo_12x4x4(energy=energy, simultaneous=sim)
    wl["settings"] = dict(wl["settings"], volume_passes=passes, poissons_ratio=0.47)
    sc = forced(ctx, wl, xcd_slabs=True, block_size=block)
    check(sc, wl, (5, 4), block)
    sc.close()


@pytest.mark.parametrize("slabs", [False, True])
@pytest.mark.parametrize("rtype", [0, 1, 2, 3])
@pytest.mark.parametrize("energy,sim", [(4, True), (7, True), (4, False), (3, True), (6, False)])
def test_damping(ctx, energy, sim, rtype, slabs):
    wl = workloads.beam_neo_12x4x4(energy=energy, simultaneous=sim)
    wl["settings"] = dict(wl["settings"], damping=0.02, rayleigh_type=rtype, pbd_damping=0.003,
                          pbd_damping_amortized=0.012)
    sc = forced(ctx, wl, xcd_slabs=slabs)
    check(sc, wl, (9, 3), 64, tick=5)
    sc.close()


@pytest.mark.parametrize("slabs", [False, True])
def test_beam_of_tiles(ctx, slabs):
    """The 96x24x24 beam, which would run as tiles, with ground and sphere."""
    wl = workloads.beam_yeoh_96x24x24()
    sc = forced(ctx, wl, xcd_slabs=slabs, block_size=256)
    check(sc, wl, (2, 1), 256)
    sc.close()


@pytest.mark.parametrize("slabs", [False, True])
def test_batch(ctx, slabs):
    """Bodies of both energies with per-tet moduli, beside each other."""
    b = workloads.boxes_batch(n_bodies=5, seed=5, cells=(2, 7))
    r = np.random.RandomState(3)
    for wl in b["bodies"][1:3]:
        wl["tet_mu"] = r.uniform(2e4, 2e6, np.asarray(wl["tets"]).size // 4).astype(np.float32)
    sc = workloads.make_batch_scene(ctx, b, xcd_slabs=slabs)
    sc.set_colour_launches()
    dt = float(b["dt"])
    sc.step(6, dt)
    assert sc.route() == (xf.ROUTE_COLOURS, 64)
    for i, wl in enumerate(b["bodies"]):
        ob = po.body_from_workload(wl, "ref64")
        ob.substep(po.params_from_settings(b["dt"], wl["settings"]), sc.order(i)[0], count=6)
        x, v = sc.get_state(i)
        assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V), i
    sc.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("cells,route", [((12, 4, 4), xf.ROUTE_BODIES), ((24, 12, 11), xf.ROUTE_TILES)])
def test_switched_between_calls(ctx, cells, route, graph):
    """The routes in turn give what either gives alone, and each call tells
    the route it took, replays of a captured call included."""
    wl = workloads.beam_yeoh(*cells, structured=False)
    dt, out = float(wl["dt"]), []
    for switch in ((0, 1, 1, 0, 0), (0, 0, 0, 0, 0), (1, 1, 1, 1, 1)):
        sc = workloads.make_scene(ctx, wl, use_graph=graph)
        assert sc.route() == (xf.ROUTE_NONE, 0)
        for on in switch:
            sc.set_colour_launches(on)
            sc.step(3, dt)
            assert sc.route()[0] == (xf.ROUTE_COLOURS if on else route)
        out.append(sc.get_state(0))
        sc.close()
    for x, v in out[1:]:
        assert np.array_equal(x, out[0][0]) and np.array_equal(v, out[0][1])


def test_route_of_a_replayed_call(ctx):
    """A call replayed from its graph after one of another route."""
    wl = workloads.beam_yeoh(12, 4, 4, structured=False)
    held = np.array([5, 9], np.uint32)
    at = np.asarray(wl["xyz"], np.float64).reshape(-1, 3)[held]
    sc = workloads.make_scene(ctx, wl, use_graph=True)
    seen = []
    for n in (2, 0, 2):
        sc.set_kinematic(0, held[:n], at[:n])
        sc.step(3, float(wl["dt"]))
        seen.append(sc.route()[0])
    sc.close()
    assert seen == [xf.ROUTE_COLOURS, xf.ROUTE_BODIES, xf.ROUTE_COLOURS]


def test_routes_of_other_modes(ctx):
    wl = workloads.beam_neo_12x4x4(energy=7)
    for opts, want in ((dict(launch_mode=xf.LAUNCH_PERSISTENT), (xf.ROUTE_PERSISTENT, 256)),
                       (dict(launch_mode=xf.LAUNCH_BLOCKS, sweep_blocks=True), (xf.ROUTE_BLOCKS, 256))):
        sc = forced(ctx, wl, **opts)
        sc.step(2, float(wl["dt"]))
        assert sc.route() == want
        sc.close()
    sc = forced(ctx, dict(wl, settings=dict(wl["settings"], energy=xf.ENERGY_CONTINUOUS_SKIN, poissons_ratio=0.45)))
    sc.step(2, float(wl["dt"]))
    assert sc.route()[0] == xf.ROUTE_RINGS
    with pytest.raises(xf.XfError):
        sc.set_colour_launches(2)
    sc.close()
