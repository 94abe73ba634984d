"""What bench.py says of the passes: only kernels that a substep launches have a time, bytes
and a bandwidth (a steady-state substep launches no sort: an empty kernel stands for it
while passes are timed), and the committed traffic of the kernels it names is found."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_the_sort_has_no_bytes_and_no_time():
    nbytes = bench.pass_bytes(1000, 10)
    assert set(nbytes) == {"p2g", "grid_update", "g2p"}
    passes = bench.pass_times({"grid_sort": (0.08, 20), "p2g": (0.8, 20), "grid_update": (0.2, 20), "g2p": (1.0, 20)},
                              nbytes)
    assert set(passes) == set(nbytes)
    assert abs(passes["g2p"]["GBps"] - nbytes["g2p"] / 50.0e-6 / 1e9) < 1e-6 and passes["p2g"]["launches"] == 20


def test_traffic_of_the_dominant_kernels_is_committed():
    for chunk in (384, 512):
        tuning = {"p2g_chunk": chunk, "g2p_threads": 256, "block_wgs": 8192}
        for workload in ("dam_break", "batched"):
            assert bench.measured_traffic(workload, "g2p", tuning) > 1e8
            assert bench.measured_traffic(workload, "p2g", tuning) > 1e7
