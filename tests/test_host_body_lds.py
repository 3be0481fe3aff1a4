"""The LDS of the single-body velocity-stepping kernel, which runs two programs
one after the other in each wave without a barrier between the waves of a
workgroup: on the CPU, every value of either program lies in its own wave's part
at 64 to 256 lanes a workgroup (a GPU run could only show an overlap by
losing the race)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_wave_uses_another_waves_lds(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "body_lds")
    p = subprocess.run([gxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "tests", "host"), "-x", "c++",
                        os.path.join(ROOT, "tests", "host", "body_lds_host_main.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stderr[-3000:]
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
