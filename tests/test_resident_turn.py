"""Turns of the launches that hold compute units (kernels/resident_turn.h): those that fit run together, the others wait in
order. Host code only, built by g++."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_resident_turn(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "resident_turn"
    b = subprocess.run([gxx, "-O1", "-std=c++17", "-pthread", f"-I{ROOT / 'alien_amd' / 'csrc'}",
                        str(ROOT / "tests" / "resident_turn_main.cpp"), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
