"""bench.py's output line without a device: short enough to be recorded whole,
with the headline untouched, each leg's numbers and its parts'; the legs in
full on stderr; the roofline from the iterations per launch that the library reports."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_line_is_short_and_legs_are_on_stderr(capsys):
    headline = {"metric": bench.METRIC, "value": 611.0, "roofline": {"kernel": "k", "frac": 0.5},
                "cpu_baseline": {"value": 2.0, "sample": "x" * 150}, "config": {"workload": "w" * 260}}
    leg = {"workload": "w" * 200, "speedup": 2.5, "iterations": 500, "ok": True,
           "per_city": [{"err": 0.1 * q, "ms": 1.0 * q} for q in range(200)],
           "cold": {"ms": 12.3456789, "note": "n" * 300, "rows": [1.0] * 300}, "stop": {"mean": {"ms": 1.0}}}
    out = dict(headline, **{k: leg for k in bench.LEG_KEYS})
    line = bench.bench_line(out)
    assert len(line) < 4000
    got = json.loads(line)
    assert {k: got[k] for k in headline} == headline
    for k in bench.LEG_KEYS:
        assert got[k] == {"speedup": 2.5, "iterations": 500, "ok": True, "cold": {"ms": 12.346}}
        assert out[k] is leg  # the caller's object stays whole
    err = capsys.readouterr().err.splitlines()
    assert [json.loads(line.split(": ", 1)[1]) for line in err] == [leg] * len(bench.LEG_KEYS)


def test_roofline_of_a_march_given_tile_fields():
    """Beyond the Infinity Cache AUTO marches whatever the colour passes' tile
    fields: half as many launches as iterations, 6.5 bytes an update."""
    res = [{"iterations": 500, "path": bench.Q.PATH_FUSED, "compressed": 1, "tile_k": 8, "tile_v": 1,
            "ms_sor": 100.0, "reserved": 2}]
    roof, _ = bench.roofline_of(res, 148_404_596, "no-such-workload", res[0]["reserved"] or None)
    assert roof["kernel"] == "k_sor_march, 2 iterations per launch" and roof["bytes_per_lup"] == 6.5
    assert roof["avg_launch_us"] == 400.0 and roof["updates_per_launch"] == 2 * 148_404_596
