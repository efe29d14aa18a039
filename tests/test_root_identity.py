"""The force loop and the h sweeps take |r_ab| and its reciprocal from one hardware estimate:
Goldschmidt's step, residual corrections of the root, Newton corrections of the reciprocal
(Markstein, IBM J. Res. Dev. 34(1), 1990).  That both come out as the IEEE sqrt and division give
them is what keeps those loops bit-identical to the general ones; this test checks it with the
host's IEEE double arithmetic and C99 fma on 4 10^6 random and adversarial operands, and that the
one exception of plain Newton corrections, a significand of all ones, is met and comes out right."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_root_and_reciprocal_are_correctly_rounded(tmp_path):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    exe = str(tmp_path / "root_check")
    subprocess.run([cc, "-O2", "-ffp-contract=off", "-std=c99",
                    os.path.join(HERE, "root_identity_check.c"), "-o", exe, "-lm"],
                   check=True, capture_output=True)
    out = subprocess.run([exe, "4000000"], check=True, capture_output=True, text=True).stdout
    assert out.strip().splitlines()[-1] == "0 0 0", out
