"""The launch levels of a sequential sweep (csrc/itnbp_graph.cpp) under the address
and undefined-behaviour sanitizers, on random graphs and sequences with repeated
messages: every position once, conflicting positions in order, each in the
earliest level, never more levels than consecutive conflict-free runs."""
import json
import os
import subprocess

from helpers import ROOT
from test_host_sanitize import ENV, GRAPH_SRC, SAN


def test_sequential_levels(tmp_path):
    exe = str(tmp_path / "levels_driver")
    src = os.path.join(ROOT, "tests", "cpp", "levels_driver.cpp")
    r = subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-Wall", "-Werror"] + SAN + [src, GRAPH_SRC, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, env=ENV, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    out = json.loads(r.stdout)
    assert out["failures"] == 0 and out["cases"] > 250 and out["shorter"] > 100, out
