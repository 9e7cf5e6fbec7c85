"""Resources of the compiled particle kernels (the compiler's own report, no GPU): where a
kernel's speed rests on two workgroups sharing a CU, its registers have to allow it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def kernels():
    from hacc_gpm_amd import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    r = subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-x", "hip", "-c",
                        os.path.join(build.CSRC, "k_particles.hip"), "-o", os.devnull,
                        "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    out, name = {}, None
    for key, val in re.findall(r"remark:.*?(Function Name|Occupancy \[waves/SIMD\]|VGPRs Spill): (\S+)", r.stderr):
        if key == "Function Name":
            name = val
        else:
            out.setdefault(name, {})[key.split()[0]] = int(val)
    return out


@pytest.mark.parametrize("kernel,n", [("k_deposit_windowsILb1E", 4), ("k_deposit_deferredILb1E", 2),
                                      ("k_bin_restILb1E", 1)])
def test_two_workgroups_per_cu(kernels, kernel, n):
    """512 threads are two waves per SIMD: two workgroups need four.  32-bit weights (Lb1)."""
    found = {k: v for k, v in kernels.items() if kernel in k}
    assert len(found) == n
    for k, v in found.items():
        assert v["Occupancy"] >= 4 and v["VGPRs"] == 0, (k, v)
