"""The appends of a block to the worklists with waves that run at different paces (tests/
append_waves.cpp, on the CPU): a wave that is late after a barrier still takes the same branch of
flush() as the others, so that no wave is left at a barrier and every cell is listed once."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("append") / "append_waves")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "c3d-2015_amd", "csrc"),
                    os.path.join(ROOT, "tests", "append_waves.cpp"), "-o", out], check=True)
    return out


# one wave pushing a tile of cells a round (the set-up) and all waves a few each (the step pass),
# with rounds enough for unforced flushes in between; late: all but the first wave, only the last,
# only the first
@pytest.mark.parametrize("late", [0b1110, 0b1000, 0b0001])
@pytest.mark.parametrize("per,rounds,pushers", [(64, 9, 1), (64, 4, 1), (8, 70, 1), (16, 35, 4)])
@pytest.mark.parametrize("every", [1, 3])
def test_waves_agree_on_the_flush(prog, per, rounds, pushers, every, late):
    r = subprocess.run([prog, str(per), str(rounds), str(pushers), str(every), str(late)],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
