"""The exact solver's shock + rarefaction root (flux64.hpp: the reference's bisection, replayed
from the root) against the bisection itself, on the host (CPU only).

Each side's function carries a rounding error of a few ulp of the speeds in it, and a face whose
|f| at some midpoint lies within that of the stopping tolerance 1e-9 may stop an iteration apart:
with speeds of order S (the pressures and densities span six decades, so S is up to 1e3 times
SPEED) a fraction of about 1e-15 S/1e-9 of the faces; there p* differs by what the tolerance
leaves, at most 1e-9/(p f'), which the replay bounds by 1e-3 and these faces by 1e-9."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("replay") / "check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                        os.path.join(ROOT, "tests", "root_replay_check.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return exe


# integer 1/gm (5/3, 7/5, 2, 3) and not (1.3, 1.1); speeds where every face replays, where the
# bend of f matters (1e-6) and where f's rounding sends faces to the plain bisection (1e3)
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 2.0, 3.0, 1.3, 1.1])
@pytest.mark.parametrize("speed", [1e-6, 1e-3, 1.0, 1e3])
def test_replay_is_the_bisection(check, gamma, speed):
    n = 20000
    r = subprocess.run([check, repr(gamma), repr(speed), str(n)], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    diff, iters, worst, _ = r.stdout.split()
    allowed = 2 + n * min(1.0, 1e-15 * 1e3 * speed / 1e-9)
    assert int(diff) <= allowed and int(iters) <= allowed, r.stdout
    assert float(worst) <= 1e-9, r.stdout
