"""The library's host side built for the CPU against the stand-in for the HIP
runtime (tests/host/): what its calls ask of the device."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCES = ["gp_runtime.cpp", "gp_plain.hip", "gp_vstep.hip", "gp_vstep_body.hip", "gp_energy.hip", "gp_terms.hip",
           "gp_xfer.hip"]


@pytest.fixture(scope="module")
def runtime_host(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("runtime_host")
    files = [os.path.join(ROOT, "gorilla-physics_amd", "csrc", s) for s in SOURCES]
    files.append(os.path.join(ROOT, "tests", "host", "runtime_host_main.cpp"))
    objs, procs = [], []
    for f in files:
        objs.append(str(d / (os.path.basename(f) + ".o")))
        procs.append(subprocess.Popen([gxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "tests", "host"), "-x", "c++",
                                       "-c", f, "-o", objs[-1]], stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                                      text=True))
    for p in procs:
        _, err = p.communicate(timeout=600)
        assert p.returncode == 0, err[-4000:]
    exe = str(d / "runtime_host")
    p = subprocess.run([gxx] + objs + ["-o", exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-4000:]
    return exe


@pytest.mark.parametrize("check", ["autotune", "device", "scratch", "staging"])
def test_host_side(runtime_host, check):
    p = subprocess.run([runtime_host, check], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
