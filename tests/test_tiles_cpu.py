"""CPU check of the lines per work-group of the sweeps (public_amd/csrc/tiles.hpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    exe = tmp_path_factory.mktemp("tiles") / "tiles_check"
    src = os.path.join(ROOT, "tests", "cpp", "tiles_check.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_tiles_fit(tiles):
    """A power of two that divides the lines side by side, in at most 512 threads."""
    for *n, d, _, lines in tiles:
        side = n[1] * n[2] if d == 0 else n[0]
        assert lines >= 1 and lines & (lines - 1) == 0 and side % lines == 0
        assert n[d] // 8 * lines <= (256 if d == 0 else 512) or lines == 1
        assert d == 0 or lines <= 16


def test_narrow_rows_only_for_more_work_groups_than_cus(tiles):
    """Along y and z a tile is as wide as it can be, or its rows are 64 bytes,
    or wider ones would leave fewer work-groups than the 256 CUs."""
    for *n, d, fp64, lines in tiles:
        if d == 0 or lines >= 8:
            continue
        wider = lines * 2
        possible = n[0] % wider == 0 and n[d] // 8 * wider <= 512
        assert not possible or n[0] * n[1] * n[2] // (n[d] * wider) < 256, (n, d, fp64, lines)


def test_cubes_keep_one_wavefront(tiles):
    got = {(tuple(n), d): lines for *n, d, fp64, lines in tiles if fp64}
    for d in range(3):
        assert got[(32, 32, 32), d] == 16
        assert got[(64, 64, 64), d] == 8
