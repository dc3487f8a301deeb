"""The walks of the bounded launches (lepic_walk.h), compiled for the host: every
node once and, for levels of up to 2^31 - 1 nodes, no step that wraps (a 32-bit
counter wraps within 262144 nodes of that bound); every cell of the sort's bricks
once, at most 2^32 threads a launch however thin the grid, and slabs and rods of
cells spread over the XCDs to 1.6 of their mean."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_node_walks(tmp_path):
    exe = tmp_path / "walk_check"
    cc = subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "walk_check.cpp"), "-o",
                         str(exe)], capture_output=True, text=True)
    if cc.returncode != 0:
        pytest.fail(cc.stderr)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "bad 0" in r.stdout, r.stdout + r.stderr
