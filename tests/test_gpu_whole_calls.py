"""Step calls of small bodies in one launch, a workgroup per body (per-colour
launch mode where every body's nodes fit the LDS of a workgroup). Bar:
bit-exact with the oracle's serial sweep in the reported order, and with the
per-colour launches that the same bodies take beside one that is too large
for LDS, at the edges of the kernel's shapes: lanes, quads, colours, the
largest body, every pass."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def separate_tets(k):
    """k unit tets 0.3 m apart along x: one colour of k tets, 4 k nodes."""
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]]
    xyz = np.concatenate([p + np.float32([0.3 * j, 0.0, 0.0]) for j in range(k)])
    return xyz.astype(np.float32).ravel(), np.arange(4 * k, dtype=np.uint32)


def body(xyz, tets, substeps=6, seed=0, **settings):
    wl = workloads.beam_neo_12x4x4()
    vel = np.random.RandomState(seed).normal(0.0, 0.2, xyz.size).astype(np.float32)
    return dict(wl, xyz=xyz, tets=tets, pinned=(xyz[0::3] == 0.0).astype(np.uint8), velocity=vel, tet_colour=None,
                substeps=substeps, settings=dict(wl["settings"], **settings))


def block(cells, **kw):
    return body(*xf.tet_block(*cells, (0.1, 0.1, 0.1), (0.0, -0.5, -0.1)), **kw)


def steps(ctx, bodies, calls=2, tick=0):
    b0 = bodies[0]
    sc = workloads.make_batch_scene(ctx, dict(bodies=bodies, dt=b0["dt"], substeps=b0["substeps"]))
    sc.set_tick(tick)
    for _ in range(calls):
        sc.step(b0["substeps"], float(b0["dt"]))
    out = [sc.get_state(i) + (sc.order(i)[0],) for i in range(len(bodies))]
    clock = (sc.time(), sc.tick())
    sc.close()
    return out, clock


def check_oracle(wl, got, calls=2, tick=0):
    ob = po.body_from_workload(wl, "ref64")
    params = po.params_from_settings(wl["dt"], wl["settings"])
    ob.tick = tick
    ob.substep(params, got[2], count=calls * wl["substeps"])
    assert np.array_equal(got[0], ob.X) and np.array_equal(got[1], ob.V)


# quads up to 64 tets a colour, one lane per tet up to 512, several tets a
# lane beyond; 640 tets fill the LDS of a workgroup, 641 take launches per colour
@pytest.mark.parametrize("k", [1, 63, 64, 65, 256, 257, 512, 513, 640, 641])
@pytest.mark.parametrize("energy", [4, 7])
def test_colour_sizes(ctx, k, energy):
    wl = body(*separate_tets(k), energy=energy, substeps=4)
    out, clock = steps(ctx, [wl])
    check_oracle(wl, out[0])
    assert clock[1] == 2 * wl["substeps"]


@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 1, 3), (12, 4, 4), (9, 9, 9)])
@pytest.mark.parametrize("nu", [0.5, 0.45])
def test_blocks_of_cells(ctx, cells, nu):
    wl = block(cells, energy=7, poissons_ratio=nu, ground_y=-0.52)
    out, _ = steps(ctx, [wl], calls=3)
    check_oracle(wl, out[0], calls=3)


PASSES = [
    dict(),
    dict(volume_passes=1),
    dict(volume_passes=2, damping=0.02, rayleigh_type=2),
    dict(damping=0.02, rayleigh_type=0),
    dict(damping=0.02, rayleigh_type=1, volume_passes=1, pbd_damping=0.003, pbd_damping_amortized=0.02),
    dict(damping=0.02, rayleigh_type=2, pbd_damping=0.003),
    dict(damping=0.02, rayleigh_type=3, pbd_damping=0.003, pbd_damping_amortized=0.02),
    dict(pbd_damping=0.003),
]


@pytest.mark.parametrize("passes", range(len(PASSES)))
@pytest.mark.parametrize("energy,sim", [(3, 1), (4, 1), (4, 0), (5, 0), (6, 1), (7, 1), (7, 0)])
def test_passes_equal_oracle_and_colour_launches(ctx, energy, sim, passes):
    """A body alone (one launch a call) and beside a body of 3,600 nodes (a
    launch per colour): the same bits, and the oracle's."""
    small = block((3, 4, 2), energy=energy, simultaneous=sim, poissons_ratio=0.45, **PASSES[passes])
    big = dict(small, **{k: v for k, v in block((24, 11, 11)).items() if k in ("xyz", "tets", "pinned", "velocity")})
    alone, clock = steps(ctx, [small], tick=5)
    both, clock_both = steps(ctx, [small, big], tick=5)
    check_oracle(small, alone[0], tick=5)
    for a, b in zip(alone[0], both[0]):
        assert np.array_equal(a, b)
    assert clock == clock_both


def test_bodies_of_different_colour_counts(ctx):
    """Bodies with 1, 6 and about 25 colours, mixed energies and different
    volume passes in one launch: each as the oracle sweeps it alone."""
    bodies = [body(*separate_tets(70), energy=4, volume_passes=1), block((1, 1, 1), energy=7, seed=1),
              block((5, 3, 4), energy=4, volume_passes=2, seed=2), block((2, 7, 3), energy=7, poissons_ratio=0.48, seed=3)]
    out, _ = steps(ctx, bodies)
    for wl, got in zip(bodies, out):
        check_oracle(wl, got)


def test_settings_state_and_pins_between_calls(ctx):
    """Settings, state, time and pins changed between whole-call steps act as
    they do on the oracle: the first-substep pin rule, unlocked pins, a
    restored state."""
    wl = block((6, 3, 3), energy=7)
    sc = xf.Scene(ctx)
    sc.add_body(wl["xyz"], wl["tets"], wl["density"], pinned=wl["pinned"], velocity=wl["velocity"],
                pin_first_substep=True)
    sc.finalize()
    big = xf.Scene(ctx)  # the same body with launches per colour
    big.add_body(wl["xyz"], wl["tets"], wl["density"], pinned=wl["pinned"], velocity=wl["velocity"],
                 pin_first_substep=True)
    other = block((24, 11, 11))
    big.add_body(other["xyz"], other["tets"], other["density"])
    big.finalize()
    dt, saved = float(wl["dt"]), []
    for s in (sc, big):
        trace = []
        for unlock, damping in ((1, 0.0), (0, 0.0), (0, 0.02), (1, 0.0)):
            for i in range(len(s.bodies)):
                s.set_settings(i, **dict(wl["settings"], unlock_pins=unlock, damping=damping, rayleigh_type=2))
            s.step(3, dt)
            trace.append(s.get_state(0))
        s.set_state(0, *trace[0])
        s.set_time(0.25)
        s.step(1, dt)
        trace.append(s.get_state(0))
        saved.append((trace, s.tick(), s.time()))
        s.close()
    for (xa, va), (xb, vb) in zip(saved[0][0], saved[1][0]):
        assert np.array_equal(xa, xb) and np.array_equal(va, vb)
    assert saved[0][1:] == saved[1][1:]
