"""The engine's host code (autotuning, plans, serving, both at once) under AddressSanitizer and UndefinedBehaviorSanitizer, linked to
a HIP runtime of host memory (tests/cpp/engine_host_test.cpp).  CPU only: no kernel is built."""

import shutil
import subprocess

import pytest

from conftest import ROOT


def test_engine_host_code_under_asan_and_ubsan(tmp_path):
    clang = shutil.which("amdclang++") or "/opt/rocm/llvm/bin/clang++"
    if not shutil.os.path.exists(clang):
        pytest.skip("clang++ not available")
    exe, csrc = tmp_path / "engine_host_test", ROOT / "fdas_amd" / "csrc"
    build = subprocess.run(
        [clang, "-x", "c++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
         f"-I{ROOT / 'include'}", f"-I{csrc}", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
         str(ROOT / "tests" / "cpp" / "engine_host_test.cpp"),
         *(str(csrc / s) for s in ("fdas_engine.cpp", "fdas_plan.cpp", "fdas_templates.cpp")), "-lpthread", "-o",
         str(exe)], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300,
                         env={"ASAN_OPTIONS": "detect_leaks=1", "UBSAN_OPTIONS": "print_stacktrace=1",
                              "PATH": "/usr/bin:/bin"})
    assert run.returncode == 0, run.stdout[-3000:] + run.stderr[-5000:]
    assert "engine host test ok" in run.stdout and "runtime error" not in run.stderr
