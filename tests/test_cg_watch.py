"""The host loop of a device CG solve (fx_cg_watch.hpp) against a scripted device: a host held up
for as long as everything queued takes is no device error, whichever kernel reports an iteration."""
import os
import subprocess

from tests.conftest import ROOT


def test_a_late_host_is_not_a_device_error(tmp_path):
    exe = tmp_path / "cg_watch"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", os.path.join(ROOT, "tests", "host", "cg_watch.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
