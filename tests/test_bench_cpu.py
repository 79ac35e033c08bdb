"""bench.py's counted traffic belongs to the tile shape that is timed."""
import glob
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def test_traffic_is_the_timed_tiles():
    import bench
    assert bench.srd_traffic([5, 5, 5]) is None
    files = glob.glob(bench.PMC_FILES)
    assert files
    for f in files:
        d = json.load(open(f))
        tile = [int(b) for b in d["command"].split("--tile ")[1].split()[:3]]
        assert bench.srd_traffic(tile) == d["kernels"]["k_srd"]["bytes_per_launch"]
    assert bench.srd_traffic([8, 4, 4]) > 1e9
