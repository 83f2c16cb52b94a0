"""The device's short division in binary32 (the precision form's build).

Inside its range the quotient equals IEEE division on every significand of the
divisor with a random, three near-midpoint, an exact and a zero numerator,
whichever neighbour of 1/d the estimate is; below it the quotient is within one
unit; outside it is NaN, which is what the one-pass sources test for.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("div32") / "division_binary32_check")
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-ffp-contract=off", os.path.join(HERE, "division_binary32_check.c"),
                    "-o", exe, "-lm"], check=True)
    return exe


@pytest.mark.parametrize("mode,step", [("range", 1), ("small", 3), ("outside", 3)])
def test_binary32(checker, mode, step):
    out = subprocess.run([checker, mode, str(step), "20241207"], check=True, capture_output=True, text=True).stdout
    samples, faults = (int(x) for x in out.split())
    assert samples > 7_000_000
    assert faults == 0
