"""bench.py without a device: the roofline from the iterations per launch that
the library reports."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_roofline_of_a_march_given_tile_fields():
    """Beyond the Infinity Cache AUTO marches whatever the colour passes' tile
    fields: half as many launches as iterations, 6.5 bytes an update."""
    res = [{"iterations": 500, "path": bench.Q.PATH_FUSED, "compressed": 1, "tile_k": 8, "tile_v": 1,
            "ms_sor": 100.0, "reserved": 2}]
    roof, _ = bench.roofline_of(res, 148_404_596, "no-such-workload", res[0]["reserved"] or None)
    assert roof["kernel"] == "k_sor_march, 2 iterations per launch" and roof["bytes_per_lup"] == 6.5
    assert roof["avg_launch_us"] == 400.0 and roof["updates_per_launch"] == 2 * 148_404_596
