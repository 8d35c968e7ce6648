"""The rows per item of a single trial's FT convolution follow the number of CUs of its device (CPU only: built with
hipcc as host code)."""

import shutil
import subprocess

import pytest

from conftest import ROOT


def test_rows_per_item_follow_the_device(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not shutil.os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe, csrc = tmp_path / "ftc_items_test", ROOT / "fdas_amd" / "csrc"
    build = subprocess.run([hipcc, "-O2", "-std=c++17", f"-I{csrc}", f"-I{ROOT / 'include'}",
                            str(ROOT / "tests" / "cpp" / "ftc_items_test.cpp"), str(csrc / "fdas_plan.cpp"),
                            str(csrc / "fdas_templates.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout[-3000:] + run.stderr[-2000:]
    assert "ftc items test ok" in run.stdout
