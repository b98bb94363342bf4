"""bench.py's roofline counts no bytes that the HBM does not move.

The bytes it attributes to each pass of a pair are at most what the counters of the committed profile
saw of that pass (profiles/traffic.json, 40^3, 46,880 record values per pair).
"""
import json
import os

import pytest

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("i,name", list(enumerate(bench.CLASS_NAMES[:3])))
def test_bytes_of_a_pass(i, name):
    with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
        seen = json.load(f)[name]
    counted = bench.record_bytes_per_pair(46880)[i]
    assert counted == seen["record_bytes_per_pair"]
    assert counted <= seen["bytes_per_pair"]
