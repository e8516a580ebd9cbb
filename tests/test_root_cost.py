"""The shock + rarefaction root of the exact solver on fast faces of a gas whose powers are not
products: Newton and a few evaluations, not the bisection's fifty (CPU only)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("gamma", [1.3, 1.1])
def test_fast_faces_take_few_powers(tmp_path, gamma):
    exe = str(tmp_path / "check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                        os.path.join(ROOT, "tests", "root_cost_check.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe, repr(gamma), "20000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    n, mean, most = r.stdout.split()
    # Newton: 10 at most and the root's own power; evaluations: midpoints within twice the
    # stopping window, which halve each time, 4 at most on either side of its edge
    assert int(n) == 20000 and float(mean) < 12.0 and int(most) <= 20, r.stdout
