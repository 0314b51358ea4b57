"""The traffic figure of the bench line belongs to the launch shape that ran."""
import json
import os
import sys

import pytest

import xpbdfem as xf

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import bench  # noqa: E402

REC = json.load(open(os.path.join(ROOT, "profiles", "traffic_beam96x24x24.json")))
BEAM = dict(n_blocks=4608, n_block_slots=906, block_lanes=64, tet_lanes=4, n_tets=331776, n_colours=24)


def test_benchmark_shape_has_a_record():
    t = bench.recorded_traffic(REC, BEAM, xf.ROUTE_BLOCKS, 256, "blocks")
    assert 10e6 < t < 14e6


@pytest.mark.parametrize("change,route,threads", [
    (dict(tet_lanes=1), xf.ROUTE_BLOCKS, 256), (dict(n_block_slots=1056), xf.ROUTE_BLOCKS, 256),
    (dict(block_lanes=128), xf.ROUTE_BLOCKS, 256), ({}, xf.ROUTE_BLOCKS, 64), ({}, xf.ROUTE_TILES, 512),
    ({}, xf.ROUTE_PERSISTENT, 256)])
def test_other_shapes_have_none(change, route, threads):
    for schedule in ("blocks", "slabs"):
        assert bench.recorded_traffic(REC, dict(BEAM, **change), route, threads, schedule) is None


def test_launches_per_colour():
    a = bench.recorded_traffic(REC, BEAM, xf.ROUTE_COLOURS, 64, "slabs")
    b = bench.recorded_traffic(REC, BEAM, xf.ROUTE_COLOURS, 64, "plain")
    assert 0 < a < b
    assert bench.recorded_traffic(REC, dict(BEAM, n_tets=1000), xf.ROUTE_COLOURS, 64, "slabs") is None
