"""Sweep-block launches with one lane per tet and more tets in a phase than a
workgroup has threads: lanes go on to further tets, whose element data,
material and energy term are loaded inside the phase. One lane per tet takes up
to 256 threads whatever block_size is, so the phases here have 257 and more
(separate tets, which all lie in one block and one phase). Bar: bit-exact with
the oracle's serial sweep in the reported order."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu

THREADS = 256
BOTH = xf.COLLIDE_GROUND | xf.COLLIDE_SPHERE


def tets(k, energy, sim=True, seed=0, **settings):
    """k separate tets above a ground plane, moving, some of them into it."""
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]]
    r = np.random.RandomState(seed)
    xyz = np.concatenate([p + np.float32([0.3 * j, 0.02 * (j % 7), 0.0]) for j in range(k)]).astype(np.float32).ravel()
    yeoh = energy in (5, 6, 7)
    st = dict(energy=energy, simultaneous=int(sim), compliance=2e-6 if yeoh else 2e-5, poissons_ratio=0.5,
              gravity=(0.0, -9.81), yeoh=(0.1095, 0.01095, 0.001095), collide=BOTH, ground_y=0.01, friction=0.4,
              sphere_c0=(3.0, 0.0, 0.0), sphere_v=(0.5, 1.0, 0.0), sphere_r=0.2)
    if energy <= 2:
        st["compliance"] = 1e-6
        st["poissons_ratio"] = 0.45
    return dict(name=f"tets{k}", xyz=xyz, tets=np.arange(4 * k, dtype=np.uint32), density=1000.0, pinned=None,
                velocity=r.normal(0.0, 0.3, xyz.size).astype(np.float32), tet_mu=None, settings=dict(st, **settings),
                dt=np.float32(1.0) / np.float32(1200.0), substeps=6)


def check(ctx, bodies, calls=(4, 2), tick=0, fused=None, **opts):
    b0 = bodies[0]
    sc = workloads.make_batch_scene(ctx, dict(bodies=bodies, dt=b0["dt"], substeps=6), sweep_blocks=True,
                                    launch_mode=xf.LAUNCH_BLOCKS, **opts)
    if fused is not None:
        assert sc.info()["fused_finish"] == int(fused)
    sc.set_tick(tick)
    for n in calls:
        sc.step(n, float(b0["dt"]))
    assert sc.route() == (xf.ROUTE_BLOCKS, THREADS) and sc.info()["tet_lanes"] == 1
    most = max(np.bincount(sc.order(i)[1]).max() for i in range(len(bodies)))
    assert most > THREADS
    for i, wl in enumerate(bodies):
        ob = po.body_from_workload(wl, "ref64")
        ob.tick = tick
        ob.substep(po.params_from_settings(wl["dt"], wl["settings"]), sc.order(i)[0], count=sum(calls))
        x, v = sc.get_state(i)
        assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V), i
    sc.close()


# one tet past the threads, a round and a remainder, exactly two rounds
@pytest.mark.parametrize("k", [257, 300, 512, 700])
@pytest.mark.parametrize("nu", [0.5, 0.47])
def test_tets_beyond_the_threads(ctx, k, nu):
    check(ctx, [tets(k, 7, poissons_ratio=nu)])


@pytest.mark.parametrize("nu", [0.5, 0.47])
@pytest.mark.parametrize("energy,sim", [(3, True), (4, True), (5, True), (6, True), (3, False), (4, False),
                                        (5, False), (6, False), (7, False), (0, True), (2, True), (12, True)])
def test_energies(ctx, energy, sim, nu):
    check(ctx, [tets(300, energy, sim, **({"poissons_ratio": nu} if energy > 2 else {}))])


@pytest.mark.parametrize("rtype", [0, 1, 2, 3])
@pytest.mark.parametrize("energy,sim,nu", [(4, True, 0.5), (7, True, 0.47), (7, False, 0.5), (5, True, 0.47)])
def test_damping(ctx, energy, sim, nu, rtype):
    check(ctx, [tets(300, energy, sim, poissons_ratio=nu, damping=0.02, rayleigh_type=rtype, pbd_damping=0.003,
                     pbd_damping_amortized=0.012)], tick=5)


def test_per_tet_moduli(ctx):
    wl = tets(300, 4, poissons_ratio=0.47)
    wl["tet_mu"] = np.random.RandomState(1).uniform(2e4, 2e6, 300).astype(np.float32)
    check(ctx, [wl])


def beam(energy, sim=True, **settings):
    wl = workloads.beam_neo_12x4x4(energy=energy, simultaneous=sim)
    return dict(wl, tet_colour=None, settings=dict(wl["settings"], **settings))


@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("energies,sim", [((7, 4), True), ((4, 7), True), ((4, 4), True), ((7, 7), True),
                                          ((3, 3), True), ((5, 5), False), ((6, 6), True)])
def test_beside_a_beam_with_the_node_phase(ctx, energies, sim, separate):
    """The tets and a beam in one scene: several launch colours, the node
    phase in the last one (or, separate, in a launch of its own), material and
    energy by tet."""
    a, b = energies
    check(ctx, [tets(260, a, sim), beam(b, sim, poissons_ratio=0.48)], fused=not separate,
          separate_finish=separate)


def test_beside_a_beam_damped(ctx):
    check(ctx, [tets(260, 7, damping=0.02, rayleigh_type=1), beam(4, damping=0.01, rayleigh_type=0)], tick=3,
          fused=False)
