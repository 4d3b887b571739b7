"""Host memory of uploads (gate calls, density matrices at chi = 32), under the address sanitizer against a HIP
runtime without a device (tests/cpp/fake_hip.hpp) whose copies run when the host waits:
every source is there, unchanged, until then."""
import json
import os
import subprocess

import pytest

from test_host_site_tasks import build_driver


@pytest.mark.parametrize("free_mib", [65536, 20])  # one launch sequence of the split pipeline; two
def test_uploads_outlive_their_copies(tmp_path, free_mib):
    exe = build_driver(tmp_path, "apply_host_driver", "-fsanitize=address")
    r = subprocess.run([exe, "20", str(free_mib)], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stderr[-3000:]
    out = json.loads(r.stdout)
    assert out["rc"] == 0 and out["changed_copies"] == 0, out
    assert out["launches"] >= (17 if free_mib > 20 else 34), out


def test_density_matrix_uploads_outlive_their_copies(tmp_path):
    exe = build_driver(tmp_path, "rdm_host_driver", "-fsanitize=address")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stderr[-3000:]
    out = json.loads(r.stdout)
    assert out["rc"] == 0 and out["changed_copies"] == 0 and out["launches"] > 10, out
