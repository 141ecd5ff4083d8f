"""Runs tests/cpp/normal_draws.hip: the device's Box-Muller functions are bit-equal to the general division,
square root and quadrant over all 2^24 arguments a draw can have (so no tolerance)."""
import subprocess

import pytest

pytestmark = pytest.mark.gpu


def test_normal_draws_exhaustive(repo):
    exe = repo / "tests" / "cpp" / "normal_draws"
    if not exe.exists():
        pytest.fail(f"{exe} not built: run dynamic-occupancy-grid-map_amd/build.py")
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
