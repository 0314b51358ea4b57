"""The plan of the tile launches on the host: it covers every colour, and
memory that runs out while planning (an allocation or a thread that fails, once
or from then on) leaves a whole plan or none, never an exception or a
terminated process, since the plan is made inside a call of the C ABI."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
EXE = os.path.join(CPP, "_build", "tile_plan_test")


def run(*args):
    if not os.path.exists(EXE):
        subprocess.run(["make", "-C", CPP, EXE], check=True, capture_output=True)
    r = subprocess.run([EXE, *map(str, args)], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, (args, r.returncode, r.stdout, r.stderr)
    return r.stdout


@pytest.mark.parametrize("cells", [(12, 7, 7), (24, 12, 11), (64, 16, 16)])
@pytest.mark.parametrize("colours", ["24", "greedy"])
def test_plan_covers_every_colour(cells, colours):
    print(run("plan", *cells, colours))


@pytest.mark.parametrize("cells,colours,step", [((12, 7, 7), "24", 1), ((24, 12, 12), "greedy", 41),
                                                ((40, 16, 16), "24", 53)])
def test_memory_that_runs_out(cells, colours, step):
    """The larger meshes plan on several threads."""
    print(run("memory", *cells, colours, step))
