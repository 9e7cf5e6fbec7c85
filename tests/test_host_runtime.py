"""The engine's control code (capi.cpp, hostcopy.cpp) on the host, against a HIP runtime
that fails where a scenario says so (tests/host/runtime_check.cpp): error paths leave a
context in a state that the next call can start from."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
GXX = shutil.which("g++")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not GXX or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("g++ or the HIP headers not available")
    out = tmp_path_factory.mktemp("runtime") / "runtime_check"
    csrc = os.path.join(ROOT, "hacc_gpm_amd", "csrc")
    srcs = [os.path.join(csrc, f) for f in ("capi.cpp", "hostcopy.cpp", "host.cpp")]
    r = subprocess.run([GXX, "-std=c++17", "-O1", "-w", "-pthread", "-D__HIP_PLATFORM_AMD__",
                        "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"), "-I", csrc, *srcs,
                        os.path.join(ROOT, "tests", "host", "runtime_check.cpp"), "-o", str(out)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return str(out)


@pytest.mark.parametrize("scenario", ["deposit", "state", "device", "unpinned", "sizes"])
def test_control_code(exe, scenario):
    r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    done, bad = (int(v) for v in r.stdout.split("\n")[-2].split())
    assert done > 0 and bad == 0, r.stdout
