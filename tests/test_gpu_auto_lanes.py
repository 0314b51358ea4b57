"""Sweep-block launches with the lanes per tet left to the library
(xf_scene_opts.tet_lanes = 0): four lanes where every launch has at most one
workgroup per compute unit and every phase fits 64 quads, else one. Bar:
bit-exact with one lane per tet and with the oracle's serial sweep in the
reported order, at the edges of the rule and of the block layout that goes
with it."""
import numpy as np
import pytest

import pyoracle as po
import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def run(ctx, wl, **opts):
    sc = workloads.make_scene(ctx, wl, sweep_blocks=True, launch_mode=xf.LAUNCH_BLOCKS, **opts)
    for _ in range(2):
        sc.step(wl["substeps"], float(wl["dt"]))
    x, v = sc.get_state(0)
    order, info = sc.order(0)[0], sc.info()
    sc.close()
    return x, v, order, info


# cells, block_lanes, settings, lanes per tet expected
CASES = [
    ((1, 1, 1), 0, {}, 4),                       # two launch colours, phases of one tet
    ((3, 2, 5), 0, {}, 4),
    ((12, 4, 4), 0, {}, 4),                      # one slot a launch, 60 tets a phase
    ((12, 4, 4), 0, dict(energy=5), 1),          # no quad form of the energy
    ((12, 4, 4), 0, dict(simultaneous=0), 1),
    ((12, 4, 4), 0, dict(damping=0.01), 1),
    ((40, 9, 11), 64, {}, 4),                    # ragged slots
    (64, 256, {}, 4),                            # one phase of 64 separate tets: every quad busy
    (65, 256, {}, 1),                            # one more than the quads
]


def mesh(cells):
    if not isinstance(cells, int):
        return xf.tet_block(*cells, (0.1, 0.1, 0.1), (0.0, -0.2, -0.2))
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]]
    xyz = np.concatenate([p + np.float32([0.3 * j, 0.0, 0.0]) for j in range(cells)])
    return xyz.astype(np.float32).ravel(), np.arange(4 * cells, dtype=np.uint32)


@pytest.mark.parametrize("cells,lanes,settings,want", CASES)
@pytest.mark.parametrize("energy", [4, 7])
def test_automatic_lanes(ctx, cells, lanes, settings, want, energy):
    wl = workloads.beam_neo_12x4x4(energy=energy)
    xyz, tets = mesh(cells)
    wl = dict(wl, xyz=xyz, tets=tets, pinned=(xyz[0::3] == 0.0).astype(np.uint8),
              settings=dict(wl["settings"], **settings))
    x, v, order, info = run(ctx, wl, block_lanes=lanes)
    assert info["tet_lanes"] == want
    ob = po.body_from_workload(wl, "ref64")
    ob.substep(po.params_from_settings(wl["dt"], wl["settings"]), order, count=2 * wl["substeps"])
    assert np.array_equal(x, ob.X) and np.array_equal(v, ob.V)


def test_automatic_lanes_packed_layout(ctx):
    """A beam whose runs of consecutive blocks would be more slots than
    compute units: the blocks are laid out so that they are not, and the
    reported order and the results are those of one lane per tet and of
    per-colour launches over the same layout."""
    wl = workloads.beam_yeoh(96, 24, 24)
    wl = dict(wl, substeps=5)
    a = run(ctx, wl)
    b = run(ctx, wl, tet_lanes=1)
    assert a[3]["tet_lanes"] == 4 and b[3]["tet_lanes"] == 1
    assert a[3]["n_block_slots"] <= 4 * 256
    assert np.array_equal(a[2], b[2])
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    sc = workloads.make_scene(ctx, wl, sweep_blocks=True)
    for _ in range(2):
        sc.step(wl["substeps"], float(wl["dt"]))
    x, v = sc.get_state(0)
    sc.close()
    assert np.array_equal(x, a[0]) and np.array_equal(v, a[1])


@pytest.mark.parametrize("dims,lanes,cap", [
    ((20, 9, 7), 192, 192),     # one slot's phases above 64 tets, few slots: runs of blocks
    ((112, 33, 31), 0, 64),     # two 64-tet slots per compute unit
    ((132, 37, 35), 0, 64),     # three, laid out to be so
    ((132, 37, 35), 200, 200),  # no multiple of the wavefront
    ((248, 60, 60), 0, 128),    # past the line of the automatic cap
])
def test_slot_caps_and_layout(ctx, dims, lanes, cap):
    """One lane per tet at the edges of the automatic slot cap and with packed
    layouts of several caps: the reported order is that of a scene of few
    large slots, and the results are those of per-colour launches."""
    wl = workloads.beam_yeoh(*dims)
    wl = dict(wl, substeps=2)
    a = run(ctx, wl, block_lanes=lanes, tet_lanes=1)
    b = run(ctx, wl, block_lanes=256, tet_lanes=1)
    assert a[3]["block_lanes"] == cap
    assert np.array_equal(a[2], b[2])
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    sc = workloads.make_scene(ctx, wl, sweep_blocks=True, block_lanes=lanes)
    for _ in range(2):
        sc.step(wl["substeps"], float(wl["dt"]))
    x, v = sc.get_state(0)
    sc.close()
    assert np.array_equal(x, a[0]) and np.array_equal(v, a[1])


@pytest.mark.parametrize("dims,lanes", [((132, 36, 36), 128), ((156, 38, 41), 192), ((172, 41, 42), 256)])
def test_workgroups_sharing_compute_units(ctx, dims, lanes):
    """Two workgroups on some compute units with phases of two, three and four
    wavefronts: the lanes that hold a phase's tets differ between them."""
    wl = workloads.beam_yeoh(*dims)
    wl = dict(wl, substeps=2)
    a = run(ctx, wl, block_lanes=lanes, tet_lanes=1)
    b = run(ctx, wl, block_lanes=64, tet_lanes=1, separate_finish=1)
    assert 256 < a[3]["n_block_slots"] / 4 <= 512
    assert all(np.array_equal(p, q) for p, q in zip(a[:3], b[:3]))


@pytest.mark.parametrize("lanes,tet_lanes", [(64, 0), (64, 4), (128, 1), (256, 1)])
@pytest.mark.parametrize("n", [3, 40])
def test_bodies_of_mixed_energies(ctx, n, lanes, tet_lanes):
    """Bodies of both energies side by side in the slots, per-tet material:
    the energy term that a lane uses is that of its tet's body."""
    wl = workloads.boxes_batch(n_bodies=n)
    dt, out = float(wl["dt"]), []
    for blocks in (True, False):
        sc = workloads.make_batch_scene(ctx, wl, sweep_blocks=True, block_lanes=lanes, tet_lanes=tet_lanes,
                                        launch_mode=xf.LAUNCH_BLOCKS if blocks else xf.LAUNCH_PER_COLOUR)
        sc.step(3, dt)
        sc.step(2, dt)
        out.append([a for i in range(n) for a in sc.get_state(i)])
        sc.close()
    assert all(np.array_equal(p, q) for p, q in zip(*out))
