"""CPU checks of the frontier kernels' lane and index arithmetic, compiled from their own header and
run by emulated workgroups (tests/emulation/lanes_check.cpp)."""
import os
import platform
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None or platform.machine() != "x86_64", reason="needs g++ on x86-64")
def test_lanes_serve_every_entry_and_neighbour_once(tmp_path):
    exe = tmp_path / "lanes_check"
    emulation = os.path.join(HERE, "emulation")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I" + emulation, "-I" + os.path.join(HERE, "..", "brook_amd", "csrc"),
                    os.path.join(emulation, "lanes_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
