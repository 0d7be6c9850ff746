"""The launches' size rules on the CPU (plast_amd/csrc/launch_rules.hpp, built with g++ into a small
checker): every launch stays below 2^32 work-items, and what one form leaves goes to another."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_launch_rules(tmp_path):
    exe = tmp_path / "launch_rules_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined",
                    f"-I{ROOT / 'plast_amd' / 'csrc'}", str(ROOT / "tests" / "launch_rules_check.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
