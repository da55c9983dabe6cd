"""The matrix-core step and the short-tile batch kernel's runs, replayed on the CPU (tests/cpp/mfma_step_emul.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("gcc") is None, reason="needs gcc and g++")
def test_step_and_short_runs_match_oracle(tmp_path):
    inc = ["-I" + os.path.join(ROOT, "mrg8_amd", "csrc"), "-I" + os.path.join(ROOT, "oracle")]
    obj, exe = str(tmp_path / "oracle.o"), str(tmp_path / "emul")
    for cmd in (["gcc", "-std=c11", "-O2", "-c", os.path.join(ROOT, "oracle", "mrg8_oracle.c"), *inc, "-o", obj],
                ["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", *inc,
                 os.path.join(ROOT, "tests", "cpp", "mfma_step_emul.cpp"), obj, "-o", exe]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("mfma step emulation ok"), r.stdout + r.stderr
