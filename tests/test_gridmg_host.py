"""Host-side parts of the multigrid solve of Regular Quad4 grids (compiled tests under tests/cpp)."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(name):
    path = os.path.join(ROOT, "tests", "cpp", "_build", name)
    if not os.path.exists(path):
        subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp"), f"_build/{name}"], check=True)
    r = subprocess.run([path], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, (r.returncode, r.stdout, r.stderr)


def test_tiles_read_lines_of_the_grid():
    run("test_gridlines")


def test_set_up_without_storage():
    run("test_gridmg_host")
