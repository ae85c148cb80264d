"""The stencil kernels' tiling (tests/tile_cover.cpp, on the CPU): every interior cell once, over
lines, sheets, small and large planes and both sides of the switch between the two orders; and
no more blocks than the cells need, but for the 1/16 of large planes and the rounding to eight."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def prog(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tile") / "tile_cover")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I",
                    os.path.join(ROOT, "c3d-2015_amd", "csrc"),
                    os.path.join(ROOT, "tests", "tile_cover.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("dims", [
    (1, 1, 1), (5000, 1, 1), (1, 5000, 1), (1, 1, 5000), (4096, 4, 4), (260, 3, 5), (7, 9, 9),
    (19, 17, 17), (2, 16, 16), (2, 257, 1), (2, 1, 255), (20, 20, 20), (3, 64, 64), (3, 4095, 1),
    (3, 4097, 1), (3, 1, 4097), (5, 65, 65), (2, 300, 301), (128, 128, 128), (61, 45, 77)])
@pytest.mark.parametrize("threads", [64, 256])
def test_each_cell_once_in_few_blocks(prog, dims, threads):
    r = subprocess.run([prog, *map(str, dims), str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    nx, ny, nz = dims
    need = -(-nx * ny * nz // threads)
    assert int(r.stdout) <= need * 17 / 16 + 8, (r.stdout, need)
