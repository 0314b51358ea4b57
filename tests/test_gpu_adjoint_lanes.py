"""Lanes per tet of the reverse sweep's colour launches: four up to 64 tets
per compute unit in a colour, one beyond. Bar: gradients bit for bit those of
the other form on the same tets."""
import numpy as np
import pytest

import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu


def separate_tets(k):
    one, t4 = xf.tet_block(1, 1, 1, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0))
    p = one.reshape(-1, 3)[t4[:4]].astype(np.float64)
    at = np.stack([0.3 * (np.arange(k) % 128), np.zeros(k), 0.3 * (np.arange(k) // 128)], 1)
    return (p[None] + at[:, None]).astype(np.float32).ravel(), np.arange(4 * k, dtype=np.uint32)


@pytest.mark.parametrize("energy", [4, 7])
@pytest.mark.parametrize("fp64", [False, True])
def test_one_and_four_lanes(ctx, energy, fp64):
    n, grads = 64 * 256, []
    r = np.random.RandomState(3)
    mu = np.exp(r.uniform(np.log(4e4), np.log(3e5), n + 1)).astype(np.float32)
    vel = r.normal(0.0, 0.3, (n + 1, 12)).astype(np.float32)
    wl = workloads.beam_fit_16x4x4()
    s = dict(wl["settings"], energy=energy, ground_y=-0.05)
    if energy == 7:
        k = xf.SKIN_YEOH[0]
        s.update(yeoh=(k, 0.1 * k, 0.01 * k), compliance=k / 1e5)
        mu = (mu / k).astype(np.float32)
    def body(first, count):
        xyz, tets = separate_tets(count)
        return dict(wl, xyz=xyz, tets=tets, pinned=(xyz[0::3] == 0.0).astype(np.uint8), settings=s, tet_colour=None,
                    tet_mu=mu[first:first + count], velocity=vel[first:first + count].ravel())

    # one colour: of n tets, with four lanes each, and with a second body's tet, with one
    for bodies in ([body(0, n)], [body(0, n), body(n, 1)]):
        sc = workloads.make_batch_scene(ctx, dict(bodies=bodies, dt=wl["dt"], substeps=4))
        target = np.concatenate([b["xyz"].astype(np.float64) for b in bodies])[None] + 0.01
        out = sc.adjoint(4, float(wl["dt"]), [4], target, window=2, fp64=fp64)
        grads.append(np.asarray(out[1]).ravel()[:n])
        sc.close()
    assert np.all(np.isfinite(grads[0])) and np.count_nonzero(grads[0]) > n // 2
    assert np.array_equal(*grads)
