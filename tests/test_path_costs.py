"""MOSP's path doubling (dyng_amd/csrc/path_costs.hpp) built for the host, a thread of the host per
workgroup (tests/native/path_costs_check.cpp): the sums of random trees, and a workgroup that gives up
its wait while the others are released."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_path_costs_on_host_threads(tmp_path):
    exe = tmp_path / "path_costs_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wno-unknown-pragmas", "-pthread",
                    "-I", str(ROOT / "tests" / "native" / "host"), "-o", str(exe),
                    str(ROOT / "tests" / "native" / "path_costs_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok ")
