"""Which repairs of several results share a launch (dyng_amd/csrc/team_rule.hpp), built for the host."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_heavy_runs_are_launched_alone(tmp_path):
    exe = tmp_path / "team_rule_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "team_rule_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=20)
    assert out.returncode == 0, out.stdout + out.stderr
