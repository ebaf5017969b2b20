"""The interval lookup of the Rys fits on the CPU: the float overload does its own bit arithmetic, so it is
held against the double one around every interval end.

The local variable leaves [-1, 1] by the rounding of T + T0, half a unit in the last place of an interval
2^-B wide: 2^(B + 1 - 24) at most, 2^-19 at B = 4 (bound 2^-18).  A float fit is ten roundings of 2^-24 on
sums of coefficients below twice the value: 1.2e-6."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_rys_intervals_in_float_and_double(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "rys_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        str(ROOT / "tests" / "host" / "rys_driver.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    vals = dict(line.split() for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines())
    for n in range(1, 8):
        assert int(vals[f"points_{n}"]) > 400 and int(vals[f"bad_{n}"]) == 0
        assert float(vals[f"smax_{n}"]) < 1.0 + 2.0 ** -18
        assert float(vals[f"err32_{n}"]) < 1.2e-6
