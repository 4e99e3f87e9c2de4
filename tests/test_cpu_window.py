"""Host check of the window order (tests/cpu_index/win_check): window, shifts and
offset of a point give the taps of the per-point kernels, inside the grid and
the window; ranges tile the order."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_index")


@pytest.fixture(scope="module")
def win_check():
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("hipcc not available")
    subprocess.check_call(["make", "-s", "-C", HERE, "win_check"])
    return os.path.join(HERE, "win_check")


# type dim ns nf0 nf1 nf2: the smallest grid allowed, odd and even sizes and widths
CASES = ["1 3 4 24 24 24", "1 3 6 24 50 37", "1 3 7 25 30 64", "1 3 13 26 27 40",
         "2 3 4 24 25 26", "2 3 6 48 24 33", "2 3 8 24 24 31", "2 3 9 25 24 30",
         "2 3 10 24 36 27", "2 3 13 28 26 30", "1 2 7 24 101 1", "2 2 10 30 24 1",
         "1 2 13 27 64 1", "2 2 6 1024 24 1"]


@pytest.mark.parametrize("case", CASES)
def test_window_check(win_check, case):
    r = subprocess.run([win_check] + case.split(), capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "OK: 0 failed checks" in r.stdout
