"""The kernels' conservative candidate tests (xdg_amd/csrc/fp32_bounds.h and
tet_contains' early rejects) on the CPU: tests/cpp/fp32_bounds_cpu.cpp
compiles the functions themselves for the host and checks each against 64-bit
or 80-bit arithmetic."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("fp32") / "fp32_bounds_cpu"
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    "-ffp-contract=off", "-I", os.path.join(ROOT, "xdg_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "fp32_bounds_cpu.cpp"), "-o", str(out)], check=True)
    return str(out)


@pytest.mark.parametrize("check", ["closest", "closest_thin", "closest_boxes", "start_boxes", "start_boxes_huge", "containment"])
def test_bound(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout == "ok\n"
