"""bench.py charges recorded hardware traffic only to a run of the kernel, batching and check
interval that were profiled, and says that it is a record."""
import pytest

import bench


@pytest.mark.parametrize("key,there", [(("sweep_nphi12", 3, 64, 2, 200), True), (("sweep_nphi12", 3, 64, 5, 200), False),
                                       (("sweep_nphi12", 3, 64, 2, 100), False), (("sweep_nphi12", 1, 64, 2, 200), False),
                                       (("sweep_spin_nphi8", 1, 64, 2, 200), True),
                                       (("sweep_spin_nphi8", 1, 16, 2, 200), False)])
def test_recorded_sweep_traffic_is_tied_to_what_was_profiled(key, there):
    traffic = bench.RECORDED_SWEEP_TRAFFIC.get(key)
    assert (traffic is not None) == there
    r = bench.roofline_rate(1000.0, traffic, 0.5)
    if there:
        assert r["frac_of"] == f"traffic recorded in {traffic[1]}"
        assert r["frac"] == pytest.approx(traffic[0] / 0.5e-3 / 1e9 / 8000.0)
    else:
        assert r["frac_of"] == "CSR bytes" and r["frac"] == pytest.approx(1000.0 / 8000.0)
