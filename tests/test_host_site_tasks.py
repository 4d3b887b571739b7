"""The tasks of the site kernel, built on the host (site_task of libitnbp.so), by a C++
driver: which messages each reads."""
import json
import os
import subprocess

from helpers import LIB, ROOT


def build_driver(tmp_path, name, *flags):
    exe = str(tmp_path / name)
    libdir = os.path.dirname(LIB)
    r = subprocess.run(["g++", "-std=c++17", "-O1", *flags, "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", name + ".cpp"),
                        "-o", exe, "-L" + libdir, "-litnbp", "-Wl,-rpath," + libdir], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_tasks_read_no_message_on_their_open_bond(tmp_path):
    r = subprocess.run([build_driver(tmp_path, "site_driver")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout)
    assert out["failures"] == 0 and out["cases"] > 1000, out
