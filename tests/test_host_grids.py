"""Launch grids of the library's host code, run against a HIP runtime without a device
(tests/cpp/fake_hip.hpp)."""
import json
import subprocess

from test_host_site_tasks import build_driver


def test_more_large_sites_than_grid_rows(tmp_path):
    """65600 sites too large for LDS in one sweep: every launch within 65535 in y and z."""
    r = subprocess.run([build_driver(tmp_path, "site_grid_driver")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout)
    assert out["path"] == "generic-f64 [vertex 65600]" and out["launches"] >= 5, out
    assert out["x"] >= 65600 and out["y"] <= 65535 and out["z"] <= 65535, out
