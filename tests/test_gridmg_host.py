"""Host-side parts of the multigrid solve of Regular Quad4 grids (compiled tests under tests/cpp)."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(name):
    path = os.path.join(ROOT, "tests", "cpp", "_build", name)
    assert os.path.exists(path), "build it first: __graft_entry__.build() (make -C tests/cpp)"
    r = subprocess.run([path], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, (r.returncode, r.stdout, r.stderr)


def test_tiles_read_lines_of_the_grid():
    run("test_gridlines")


def test_set_up_without_storage():
    run("test_gridmg_host")
