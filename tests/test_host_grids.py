"""Launch grids of the library's host code, run against a HIP runtime without a device
(tests/cpp/fake_hip.hpp)."""
import json
import subprocess

import pytest

from test_host_site_tasks import build_driver


def test_more_large_sites_than_grid_rows(tmp_path):
    """65600 sites too large for LDS in one sweep: every launch within 65535 in y and z."""
    r = subprocess.run([build_driver(tmp_path, "site_grid_driver")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout)
    assert out["path"] == "generic-f64 [vertex 65600]" and out["launches"] >= 5, out
    assert out["x"] >= 65600 and out["y"] <= 65535 and out["z"] <= 65535, out


@pytest.mark.parametrize("a,b", [(3, 3), (4, 5), (5, 5), (5, 6), (5, 7), (6, 6), (6, 7), (7, 7), (7, 8), (3, 33), (3, 34),
                                 (8, 8), (9, 9)])
def test_fp64_rotations_share_the_device_evenly(tmp_path, a, b):
    """The chi = 32 FP64 sweep's rotations: 256 units of work per degree-4 site, of which
    no workgroup takes more than an even share of the 512 resident ones (two per CU), or
    than a 64th of a site where there are fewer units than that."""
    r = subprocess.run([build_driver(tmp_path, "eig_split_driver"), str(a), str(b)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout)
    sites, wgs = (a - 2) * (b - 2), out["workgroups"]
    assert out["rc"] == 0 and 0 < wgs <= 512, out
    assert -(-256 * sites // wgs) <= max(-(-256 * sites // 512), 4), (sites, wgs)
