"""CPU model of the end of a synchronous call (vkhel_amd/csrc/call_wait.h):
tests/c/call_wait_model.cpp runs the library's own wait with a stand-in for
the device.  A call returns only after its work is done, also where the
kernel that marks its completion could not be launched, and it watches that
kernel's word only in a run of calls that the program does not follow by
synchronising the device."""
import os
import subprocess

from vkhel_amd import lib as L

SRC = os.path.join(L.REPO, "tests", "c", "call_wait_model.cpp")


def test_call_wait_model(tmp_path):
    exe = tmp_path / "call_wait_model"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror",
                    "-I", os.path.join(L.REPO, "vkhel_amd", "csrc"), SRC,
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("model ok")
