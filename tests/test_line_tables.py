"""The front end makes the twiddle tables that its transforms read, once each, and no others (CPU only: built with
hipcc as host code)."""

import shutil
import subprocess

import pytest

from conftest import ROOT


def test_tables_of_every_length(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not shutil.os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe, csrc = tmp_path / "line_tables_test", ROOT / "fdas_amd" / "csrc"
    build = subprocess.run([hipcc, "-O2", "-std=c++17", f"-I{csrc}", f"-I{ROOT / 'include'}",
                            str(ROOT / "tests" / "cpp" / "line_tables_test.cpp"), str(csrc / "fdas_plan.cpp"),
                            str(csrc / "fdas_templates.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout[-3000:] + run.stderr[-2000:]
    assert "line tables test ok" in run.stdout
