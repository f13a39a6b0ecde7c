"""The C ABI's host code on its own: csrc/bmx_capi.hip compiled for the host
only and run over a simulated device (tests/host/capi_host.cpp) that keeps
which buffers the executed launches left current.  Covers what no device run
can force: the bookkeeping after operations that fail."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "boltzmannmfx_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    from boltzmannmfx_amd import build
    out = tmp_path_factory.mktemp("host")
    obj, exe = str(out / "capi_host.o"), str(out / "capi_host")
    subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-O0",
                    "-std=c++17", "-x", "hip", "-I" + os.path.join(ROOT, "include"),
                    "-I" + CSRC, "-c", os.path.join(ROOT, "tests", "host", "capi_host.cpp"),
                    "-o", obj], check=True)
    # the HIP runtime is simulated; launches that no case reaches stay undefined
    subprocess.run(["g++", "-no-pie", "-Wl,--unresolved-symbols=ignore-all", obj, "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("case", ["graph_with_chem", "failed_capture", "failed_build",
                                  "adjoint_error", "tile_follows_reach"])
def test_bookkeeping_matches_the_launches(exe, case):
    p = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
