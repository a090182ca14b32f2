"""The tracked counter file answers for the passes the tracked bench line timed
(the bench takes its roofline's traffic from it by pass and direction)."""
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_of_every_timed_pass():
    line = json.loads(open(os.path.join(ROOT, "profiles", "launch_tgv256.json")).readline())
    kernels = json.load(open(os.path.join(ROOT, "profiles", "traffic_tgv256.json")))["kernels"]
    assert set(line["kernels_ms_per_launch"]) == set(kernels)
    for name, k in kernels.items():
        assert k["bytes_per_launch"] == k["read_bytes"] + k["write_bytes"] > 8 * 257 ** 3, name
    # counters of two runs agree to a few tenths of a per cent
    dominant = kernels[line["roofline"]["kernel"].replace(" (", "_").rstrip(")")]
    assert abs(line["roofline"]["traffic"] / dominant["bytes_per_launch"] - 1.0) < 0.02
