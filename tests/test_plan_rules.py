"""The work plans of ensembles on the host (CPU), with the functions that the
device plans with (gravidy_amd/csrc/h4_kernels.hpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
def test_plans_of_ensembles(tmp_path):
    exe = tmp_path / "plan_rules"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "--offload-arch=gfx950",
                    "-I", os.path.join(ROOT, "gravidy_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan_rules.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "plan rules ok" in proc.stdout
