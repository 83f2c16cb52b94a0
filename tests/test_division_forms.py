"""The device's division without scaling and without selects equals IEEE division.

recip() refines an estimate of 1/d by two Newton steps; rdiv() corrects
q0 = RN(a r) by its exact remainder, formed so that a vanishing one keeps q0, a
zero of either sign included.  Checked in binary64 against a / d on random
operands, quotients next to a rounding midpoint, exact quotients and signed
zeros, for estimates good to 24 bits and to 28 bits.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("div") / "division_forms_check")
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-ffp-contract=off", os.path.join(HERE, "division_forms_check.c"),
                    "-o", exe, "-lm"], check=True)
    return exe


@pytest.mark.parametrize("bits", [24, 28])
def test_division_equals_ieee(checker, bits):
    out = subprocess.run([checker, "1500000", "20241207", str(bits)], check=True, capture_output=True, text=True).stdout
    samples, bad = (int(x) for x in out.split())
    assert samples == 9_000_000
    assert bad == 0
