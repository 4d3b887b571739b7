"""Launch sequences of a gate call on the split pipeline, planned on the host against a
HIP runtime without a device (tests/cpp/fake_hip.hpp)."""
import json
import subprocess

from test_host_site_tasks import build_driver


def run(exe, gates, free_mib):
    r = subprocess.run([exe, str(gates), str(free_mib)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout)
    assert out["rc"] == 0, out
    return out


def test_sequences_fit_half_the_free_memory(tmp_path):
    """17 launches a sequence and 2 around the call; the workspace is the largest buffer."""
    exe = build_driver(tmp_path, "apply_host_driver")
    for gates, free_mib, sequences in ((20, 65536, 1), (20, 20, 2), (57, 64, 2), (200, 100, 4), (20, 3, 20)):
        out = run(exe, gates, free_mib)
        assert out["launches"] == 17 * sequences + 2, (gates, free_mib, out)
        if sequences < 20:
            assert out["largest_alloc"] <= free_mib << 19, (gates, free_mib, out)


def test_planning_is_linear_in_the_gates(tmp_path):
    """Eight times the gates take about eight times as long (fifty with a plan of the
    whole sequence per gate)."""
    exe = build_driver(tmp_path, "apply_host_driver")
    few, many = (min(run(exe, n, 65536)["us"] for _ in range(3)) for n in (500, 4000))
    assert many <= 24 * few, (few, many)
