"""Memory rules of the served form on the CPU: pk_server.cpp linked with a
device that is a number of bytes and a context whose steps take as many of
them as the job says (tests/cpp/server_memory_test.cpp)."""
from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def server_bin(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("server") / "server_memory_test")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           f"-I{os.path.join(ROOT, 'include')}", "-Wno-deprecated-declarations",
                           os.path.join(ROOT, "tests", "cpp", "server_memory_test.cpp"),
                           os.path.join(ROOT, "pakman_plus_amd", "csrc", "pk_server.cpp"), "-lpthread", "-o", out])
    return out


@pytest.mark.parametrize("case", ["cutoff", "nodes"])
def test_later_steps_get_the_kept_blocks(server_bin, case):
    """A cutoff or macro nodes short of memory get the blocks of released jobs
    back, as a count does."""
    r = subprocess.run([server_bin, case], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout.strip()) == (0, "ok"), r.stdout + r.stderr


def test_release_without_host_memory(server_bin):
    """A release that can allocate nothing on the host neither throws through the
    C entry nor loses the result block."""
    r = subprocess.run([server_bin, "release"], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout.strip()) == (0, "ok"), r.stdout + r.stderr
