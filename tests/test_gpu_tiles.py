"""Several colours of a sweep in one launch, a workgroup per tile of nodes
(per-colour launch mode, scenes whose bodies are not swept whole in a
workgroup). Bar: bit-exact with the oracle's serial sweep in the reported
order and with the persistent launch of the same scene, at the edges of the
kernel's shapes: tiles, spans, lanes, own nodes, step calls of every parity."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def block(cells, structured=False, seed=0, scale=0.1, **settings):
    wl = workloads.beam_yeoh(*cells, structured=structured)
    vel = np.random.RandomState(seed).normal(0.0, 0.2, np.asarray(wl["xyz"]).size).astype(np.float32)
    return dict(wl, velocity=vel, settings=dict(wl["settings"], **settings))


def scene(ctx, bodies, **opts):
    b0 = bodies[0]
    return workloads.make_batch_scene(ctx, dict(bodies=bodies, dt=b0["dt"], substeps=b0["substeps"]), **opts)


def states(sc, n):
    return [a for i in range(n) for a in sc.get_state(i)]


def tiled(sc, dt):
    """Whether a step call takes fewer launches than colours."""
    return sc.profile(2, dt)[2] < 2 * sc.info()["n_colours"]


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


# cells, the caller's 24 colours or greedy ones; the first is the smallest
# whose tiles are the choice, the last has more own nodes per tile than a
# workgroup has lanes and phases of several tets a lane
@pytest.mark.parametrize("cells,structured", [((16, 8, 8), False), ((16, 8, 8), True), ((23, 11, 13), False),
                                              ((40, 16, 15), True), ((70, 21, 19), False)])
@pytest.mark.parametrize("energy,sim", [(4, 1), (7, 1), (4, 0), (7, 0), (3, 1), (5, 0), (6, 1)])
def test_equals_persistent(ctx, cells, structured, energy, sim):
    if energy not in (4, 7) and cells != (23, 11, 13):
        pytest.skip("one mesh for the rarer energies")
    wl = block(cells, structured, energy=energy, simultaneous=sim, poissons_ratio=0.47)
    dt, out = float(wl["dt"]), []
    for mode in (xf.LAUNCH_PER_COLOUR, xf.LAUNCH_PERSISTENT):
        sc = scene(ctx, [wl], launch_mode=mode)
        for n in (1, 2, 3, 2):
            sc.step(n, dt)
        out.append(states(sc, 1) + [sc.order(0)[0], np.float32([sc.time(), sc.tick()])])
        if mode == xf.LAUNCH_PER_COLOUR:
            assert tiled(sc, dt)
        sc.close()
    assert same(*out)


def test_large_tiles_equal_persistent(ctx):
    """160,000 nodes: more own nodes per tile than lanes, spans of few colours."""
    wl = block((126, 35, 34))
    dt, out = float(wl["dt"]), []
    for mode in (xf.LAUNCH_PER_COLOUR, xf.LAUNCH_PERSISTENT):
        sc = scene(ctx, [wl], launch_mode=mode)
        sc.step(3, dt)
        out.append(states(sc, 1))
        if mode == xf.LAUNCH_PER_COLOUR:
            assert tiled(sc, dt)
        sc.close()
    assert same(*out)


@pytest.mark.parametrize("energy", [4, 7])
def test_equals_oracle(ctx, energy):
    wl = block((16, 9, 8), energy=energy)
    sc = scene(ctx, [wl])
    sc.step(3, float(wl["dt"]))
    sc.step(2, float(wl["dt"]))
    ob = po.body_from_workload(wl, "ref64")
    ob.substep(po.params_from_settings(wl["dt"], wl["settings"]), sc.order(0)[0], count=5)
    x, v = sc.get_state(0)
    sc.close()
    assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V)


def test_bodies_of_many_sizes(ctx):
    """Bodies from one cell to several tiles, mixed energies and per-tet
    moduli, beside each other."""
    bodies = [block((24, 12, 11), energy=7), block((1, 1, 1), energy=4, seed=1), block((9, 6, 5), energy=4, seed=2),
              block((3, 2, 2), energy=7, poissons_ratio=0.48, seed=3), block((30, 10, 10), energy=7, seed=4)]
    dt, out = float(bodies[0]["dt"]), []
    mu = [np.random.RandomState(9).uniform(2e4, 2e6, len(b["tets"]) // 4 if np.asarray(b["tets"]).ndim == 1 else
                                           len(b["tets"])).astype(np.float32) for b in bodies]
    for mode in (xf.LAUNCH_PER_COLOUR, xf.LAUNCH_PERSISTENT):
        sc = scene(ctx, bodies, launch_mode=mode)
        sc.step(3, dt)
        got = states(sc, 5)
        sc.set_tet_mu(0, mu[0])  # the material of the tiles follows
        sc.set_tet_mu(3, mu[3])
        sc.step(2, dt)
        got += states(sc, 5)
        sc.set_settings(4, **dict(bodies[4]["settings"], compliance=3e-6))
        sc.step(1, dt)
        got += states(sc, 5)
        if mode == xf.LAUNCH_PER_COLOUR:
            assert tiled(sc, dt)
        out.append(got)
        sc.close()
    assert same(*out)


def test_changes_between_calls(ctx):
    """Passes and held nodes come and go between step calls (colour launches
    while they are there), states are set and read, graph or not."""
    wl = block((17, 9, 8))
    dt, out = float(wl["dt"]), []
    held = np.arange(5, 60, 7, dtype=np.uint32)
    at = np.asarray(wl["xyz"], np.float64).reshape(-1, 3)[held] + 0.01
    for graph in (True, False):
        sc = scene(ctx, [wl], use_graph=graph)
        trace = []
        for damping, kin, n in ((0.0, False, 3), (0.02, False, 2), (0.0, True, 3), (0.0, False, 1), (0.0, False, 1)):
            sc.set_settings(0, **dict(wl["settings"], damping=damping, rayleigh_type=2))
            sc.set_kinematic(0, held if kin else held[:0], at if kin else at[:0])
            sc.step(n, dt)
            trace += states(sc, 1)
            if len(trace) == 2:
                t3 = sc.time()
        assert tiled(sc, dt)
        sc.set_state(0, *trace[:2])
        sc.set_time(t3)
        sc.step(2, dt)
        trace += states(sc, 1)
        out.append(trace)
        sc.close()
    assert same(*out)
    # the first three substeps and the ones after the restore, on the oracle
    # (nodes that were held keep the zero inverse mass they were given)
    ob = po.body_from_workload(wl, "ref64")
    sc = scene(ctx, [wl])
    order = sc.order(0)[0]
    sc.close()
    ob.substep(po.params_from_settings(wl["dt"], dict(wl["settings"])), order, count=3)
    assert np.array_equal(out[0][0], ob.X) and np.array_equal(out[0][1], ob.V)
    ob.w[held] = 0.0
    ob.substep(po.params_from_settings(wl["dt"], dict(wl["settings"])), order, count=2)
    assert np.array_equal(out[0][-2], ob.X) and np.array_equal(out[0][-1], ob.V)
