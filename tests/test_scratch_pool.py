"""The pool of the applies' scratch (dyng_amd/csrc/scratch_pool.hpp), built for the host, plain and with
AddressSanitizer."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("sanitize", [False, True], ids=["plain", "asan"])
def test_scratch_pool(tmp_path, sanitize):
    exe = tmp_path / "scratch_pool_check"
    extra = ["-g", "-fsanitize=address", "-fno-omit-frame-pointer"] if sanitize else []
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", *extra, "-o", str(exe),
                    str(ROOT / "tests" / "native" / "scratch_pool_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
