"""The library's host code without a GPU: host_logic.hip (launches, their arguments,
what is left behind where memory runs out) on the host-memory HIP runtime of
fake_hip.cpp, which the test program defines in place of the real one's symbols."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = shutil.which("hipcc") or os.path.join(ROCM, "bin", "hipcc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("host_logic")
    lib = os.path.join(ROOT, "gpue_amd")
    out = str(d / "host_logic")
    for cmd in (
        [HIPCC, "-std=c++17", "-O1", "-fPIC", "-x", "hip", "--offload-host-only", "-I" + os.path.join(ROOT, "include"),
         "-c", os.path.join(HERE, "host", "host_logic.hip"), "-o", str(d / "logic.o")],
        ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
         "-c", os.path.join(HERE, "host", "fake_hip.cpp"), "-o", str(d / "fake.o")],
        ["g++", str(d / "logic.o"), str(d / "fake.o"), "-o", out, "-L" + lib, "-lgpue_amd", "-Wl,-rpath," + lib,
         "-Wl,-rpath-link," + os.path.join(ROCM, "lib"), "-pthread"],
    ):
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
    return out


@pytest.mark.parametrize("check", ["batch_norms", "batch_members_change", "field_out_of_memory", "pinned_memory",
                                   "step_blocks", "line_runs", "line_reports", "service_captures", "tuner_fails", "tuner_times_steps",
                                   "tuner_regroups", "batch_boxes"])
def test_host_logic(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-2000:]
