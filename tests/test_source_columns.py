"""The one-pass sources' lanes stay on their ring and inside the arrays.

A wave holds 64 columns whatever the ring's length, so on short rings most of
its lanes lie past the ring's end.  Every index is gone through on the host, for
every ring length up to and past two waves' cells.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("columns") / "source_columns_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "source_columns_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("energy", [0, 1])
@pytest.mark.parametrize("ny", [4, 33])
def test_every_index(checker, ny, energy):
    for nx in range(1, 131):
        out = subprocess.run([checker, str(nx), str(ny), str(energy)], check=True, capture_output=True, text=True).stdout
        cells, faults = (int(x) for x in out.split())
        assert (cells, faults) == (nx, 0), (nx, ny, energy)
