"""The workgroup size that the autotuner reports: one it compared, where the
launches take it, and the caller's where they choose their own (whole calls,
tiles, blocks with one lane per tet)."""
import pytest

import workloads
import xpbdfem as xf

pytestmark = pytest.mark.gpu

CALLERS = 192  # not among the sizes the tuner tries


def tuned(ctx, wl, colours=False, **opts):
    sc = workloads.make_scene(ctx, wl, block_size=CALLERS, **opts)
    sc.set_colour_launches(colours)
    mode, size, ms = sc.autotune(4, float(wl["dt"]), reps=2)
    assert ms > 0.0
    sc.step(2, float(wl["dt"]))
    route, threads = sc.route()
    lanes = sc.info()["tet_lanes"]
    sc.close()
    return mode, size, route, threads, lanes


@pytest.mark.parametrize("cells,want", [((12, 4, 4), xf.ROUTE_BODIES), ((40, 16, 15), xf.ROUTE_TILES)])
def test_routes_with_a_size_of_their_own(ctx, cells, want):
    mode, size, route, _, _ = tuned(ctx, workloads.beam_yeoh(*cells))
    assert (mode, size, route) == (xf.LAUNCH_PER_COLOUR, CALLERS, want)


def test_colour_launches(ctx):
    mode, size, route, threads, _ = tuned(ctx, workloads.beam_yeoh(40, 16, 15), colours=True)
    if mode == xf.LAUNCH_PER_COLOUR:
        assert route == xf.ROUTE_COLOURS and size == threads and size in (64, 128, 256)


def test_blocks_of_one_lane(ctx):
    """The serial solve has no form with four lanes per tet."""
    wl = workloads.beam_yeoh(24, 8, 8)
    wl["settings"] = dict(wl["settings"], simultaneous=0)
    mode, size, route, _, lanes = tuned(ctx, wl, colours=True, sweep_blocks=True)
    assert (mode, size, route, lanes) == (xf.LAUNCH_BLOCKS, CALLERS, xf.ROUTE_BLOCKS, 1)


def test_blocks_of_four_lanes(ctx):
    mode, size, route, threads, lanes = tuned(ctx, workloads.beam_yeoh(24, 8, 8), colours=True, sweep_blocks=True)
    assert (mode, route) == (xf.LAUNCH_BLOCKS, xf.ROUTE_BLOCKS)
    assert (size == threads and size in (64, 128, 256)) if lanes == 4 else size == CALLERS
