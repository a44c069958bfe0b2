"""Device memory under a limit (tests/consumers/device_memory.cpp, built here with
HIP calls that only count bytes; no GPU)."""
import glob
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("memory") / "device_memory")
    csrc = os.path.join(ROOT, "tbsla_amd", "csrc")
    src = [os.path.join(ROOT, "tests", "consumers", "device_memory.cpp"), os.path.join(csrc, "device", "mirror.cpp")]
    src += sorted(glob.glob(os.path.join(csrc, "host", "*.cpp"))) + glob.glob(os.path.join(csrc, "device", "runspace.cpp"))
    # (what the mirrors do not call, the products and the engines, is left undefined)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-o", exe, *src, "-lpthread",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return exe


@pytest.mark.parametrize("what", ["mirror", "spaces"])
def test_memory(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
