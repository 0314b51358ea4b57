"""The adjoint of small bodies with a checkpoint window per launch. Bar: loss,
per-body loss and gradients equal, bit for bit, those of the launches per
colour (the allocation-free entry point, and the same bodies beside one that
is too large for a workgroup's LDS), at the edges of the kernels' shapes."""
import numpy as np
import pytest

import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def separate_tets(k):
    """k unit tets 0.3 m apart along x: one colour of k tets, 4 k nodes."""
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]]
    xyz = np.concatenate([p + np.float32([0.3 * j, 0.0, 0.0]) for j in range(k)])
    return xyz.astype(np.float32).ravel(), np.arange(4 * k, dtype=np.uint32)


def body(xyz, tets, energy, seed=0, ground=-0.05, nu=0.5):
    wl = workloads.beam_fit_16x4x4()
    r = np.random.RandomState(seed)
    k = xf.SKIN_YEOH[0]
    mu = np.exp(r.uniform(np.log(4e4), np.log(3e5), tets.size // 4)).astype(np.float32)
    s = dict(wl["settings"], energy=energy, ground_y=ground, poissons_ratio=nu)
    if energy == 7:
        s.update(yeoh=(k, 0.1 * k, 0.01 * k), compliance=k / 1e5)
        mu = (mu / k).astype(np.float32)
    return dict(wl, xyz=xyz, tets=tets, pinned=(xyz[0::3] == 0.0).astype(np.uint8), tet_mu=mu, tet_colour=None,
                velocity=r.normal(0.0, 0.3, xyz.size).astype(np.float32), settings=s)


def adjoint(ctx, bodies, substeps, window, loss_at, **kw):
    sc = workloads.make_batch_scene(ctx, dict(bodies=bodies, dt=bodies[0]["dt"], substeps=substeps))
    rest = np.concatenate([b["xyz"].astype(np.float64) for b in bodies])
    targets = np.stack([rest + 0.01 * (j + 1) for j in range(len(loss_at))])
    if kw.get("noalloc"):
        sc.step(1, float(bodies[0]["dt"]))  # the per-tet material storage
        for i, b in enumerate(bodies):
            sc.set_state(i, b["xyz"].astype(np.float64), b["velocity"].astype(np.float64))
        sc.set_time(0.0)
    out = sc.adjoint(substeps, float(bodies[0]["dt"]), loss_at, targets, window=window, per_body=True, **kw)
    states = [sc.get_state(i) for i in range(len(bodies))]
    clock = sc.time()
    sc.close()
    return out, states, clock


def same(a, b):
    (la, ga, ba), sa, ca = a
    (lb, gb, bb), sb, cb = b
    assert la == lb and ca == cb
    assert np.array_equal(ga, gb) and np.array_equal(ba, bb)
    assert np.all(np.isfinite(ga)) and np.any(ga != 0.0)
    for (xa, va), (xb, vb) in zip(sa, sb):
        assert np.array_equal(xa, xb) and np.array_equal(va, vb)


# one-lane and quad phases of both sweeps: 64 and 128 tets a colour, then one
# lane per tet to 512 and beyond; 640 fill the LDS
@pytest.mark.parametrize("k", [1, 64, 65, 128, 129, 512, 513, 640])
@pytest.mark.parametrize("energy", [4, 7])
def test_colour_sizes(ctx, k, energy):
    b = [body(*separate_tets(k), energy)]
    args = (ctx, b, 7, 3, [2, 3, 7])
    same(adjoint(*args), adjoint(*args, noalloc=True))


@pytest.mark.parametrize("window,loss_at", [(1, [5]), (4, [1, 2, 3, 4, 9]), (9, [9]), (50, [3, 9])])
@pytest.mark.parametrize("nu", [0.5, 0.45])
def test_windows_and_losses(ctx, window, loss_at, nu):
    """Windows of one substep, a ragged last window, a single window; losses
    inside, at and beside window ends; contact with friction from the start."""
    cells = xf.tet_block(5, 3, 4, (0.1, 0.1, 0.1), (0.0, -0.05, 0.0))
    args = (ctx, [body(*cells, 7, ground=-0.048, nu=nu)], 9, window, loss_at)
    same(adjoint(*args), adjoint(*args, noalloc=True))


@pytest.mark.parametrize("fp64", [False, True])
def test_beside_a_large_body(ctx, fp64):
    """Three bodies of different colour counts and energies, alone (windows)
    and beside a body of 3,600 nodes (launches per colour)."""
    blk = lambda c: xf.tet_block(*c, (0.1, 0.1, 0.1), (0.0, -0.05, 0.0))  # noqa: E731
    small = [body(*blk((4, 3, 3)), 4, 1), body(*separate_tets(70), 7, 2), body(*blk((1, 1, 1)), 4, 3)]
    big = body(*blk((24, 11, 11)), 7, 4)
    a = adjoint(ctx, small, 8, 3, [3, 8], fp64=fp64)
    b = adjoint(ctx, small + [big], 8, 3, [3, 8], fp64=fp64)
    n = a[0][1].size
    assert np.array_equal(a[0][1], b[0][1][:n]) and np.array_equal(a[0][2], b[0][2][:3])
    assert np.any(a[0][1] != 0.0) and a[2] == b[2]
    for (xa, va), (xb, vb) in zip(a[1], b[1]):
        assert np.array_equal(xa, xb) and np.array_equal(va, vb)


@pytest.mark.parametrize("k", [64, 65, 256, 257])
def test_fp64_colour_sizes(ctx, k):
    blk = xf.tet_block(24, 11, 11, (0.1, 0.1, 0.1), (0.0, -0.05, 0.0))
    b = body(*separate_tets(k), 7)
    a = adjoint(ctx, [b], 5, 2, [2, 5], fp64=True)
    both = adjoint(ctx, [b, body(*blk, 7, 4)], 5, 2, [2, 5], fp64=True)
    assert np.array_equal(a[0][1], both[0][1][:k]) and a[0][2][0] == both[0][2][0]
    assert np.any(a[0][1] != 0.0)
