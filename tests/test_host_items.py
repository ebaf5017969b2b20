"""The cutting of ket lists into work items and the kernels' walk over them, on the CPU under
AddressSanitizer: every ket of a bra with every one of the bra's primitive pairs exactly once, inside the
bra's segments, for every number of lanes per ket."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_work_items_cover_each_ket_once(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "items_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=undefined", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        str(ROOT / "tests" / "host" / "items_driver.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stderr[-4000:]
    vals = dict(line.split() for line in run.stdout.splitlines())
    assert int(vals["kets"]) > 10 ** 6
    assert all(int(vals[k]) == 0 for k in ("bad_cover", "bad_segment", "bad_pack"))
