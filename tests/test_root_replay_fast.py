"""The replayed bisection (shock_raref_root of flux64.hpp) where speeds near 1e4 send faces to the
plain bisection: few faces may stop an iteration apart (CPU only)."""
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


# Speeds of 1 to 1e6: a face replays where |du| + c2 is below 1e4, and there f's rounding (about
# 1e-16 of the speeds) can move the stop where |f| lies within it of 1e-9: a fraction of up to
# 1e-16 * 1e4 / 1e-9 = 1e-3 of the few midpoints next to the stop.  An edge of the stopping window
# that is 10% off moves 2% of the faces.
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 2.0, 3.0, 1.3, 1.1])
def test_few_faces_stop_apart(check, gamma):
    n = 20000
    r = subprocess.run([check, repr(gamma), "1000.0", str(n)], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr
    diff, iters, worst, _ = r.stdout.split()
    assert int(diff) <= 0.01 * n and int(iters) <= 0.01 * n, r.stdout
    assert float(worst) <= 1e-9, r.stdout
