"""The host's bounds of a paged batch's chunks against the rule that the device
evaluates over the lengths (molot_amd/csrc/paged_plan.hpp), exhaustively over a
lone sequence's lengths (CPU: the header is plain C++)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_chunks_within_the_plan(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path / "paged_plan_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror",
                    os.path.join(HERE, "cpp", "paged_plan_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
