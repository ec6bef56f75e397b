"""Turns at a device's CUs for launches whose workgroups wait for one another
(host/resident_gate.h, compiled here with the host compiler, also under
ThreadSanitizer)."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("flags", [[], ["-fsanitize=thread", "-static-libtsan"]])
def test_turns(tmp_path, flags):
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "gate")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Werror", "-pthread", *flags,
                    "-I" + os.path.join(PKG, "host"), os.path.join(HERE, "plan", "gate_driver.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe] + (["untimed"] if flags else []), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "gate: ok" in r.stdout, (r.returncode, r.stdout + r.stderr)
