"""The host threads that copy a large call's data (s2tc_amd/csrc/staging.h): tests/crew_checks.cpp."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copy_crew(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = str(tmp_path / "crew_checks")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", "-I", os.path.join(ROOT, "s2tc_amd", "csrc"),
                    "-o", exe, os.path.join(ROOT, "tests", "crew_checks.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
