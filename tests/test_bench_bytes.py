"""bench.py's algorithmic bytes of a kernel are what it cannot do without, so
no kernel moves fewer by the committed counters, in either precision."""
import json
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

TRAFFIC = json.load(open(os.path.join(ROOT, "profiles", "traffic.json")))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_algorithmic_bytes_are_moved(prec):
    import bench
    for kernel, moved in TRAFFIC[prec].items():
        need = bench.kernel_bytes(kernel, 9, True, 128, prec)
        assert 0 < need <= moved, (kernel, need, moved)
