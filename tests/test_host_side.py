"""The handle's host side on the CPU, where memory is refused and where it
keeps what the device owns: host_harness.cpp holds su2hip_api.cpp with a runtime
whose allocations can fail and kernels that only record their launches."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("harness") / "host_harness")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(HERE, "host_harness.cpp"), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all", "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("scenario", [
    "refused_buffers",
    "refused_call",
    "refused_tables",
    "refused_growth",
    "budget_requests",
    "weight_keeps_draws",
    "added_lattice_sweeps",
    "fetch_waits_idle",
    "many_alike",
    "failed_launch",
    "which_sweeps_pair",
])
def test_host_side(harness, scenario):
    r = subprocess.run([harness, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
