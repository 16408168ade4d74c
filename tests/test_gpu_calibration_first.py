"""The first calibration of a process."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TWICE = """
from cswap_amd import swap
e = swap.SwapEngine(pinned_bytes=256 << 20, device_bytes=64 << 20)
print(e.calibrate().probe_latency_us, e.calibrate().probe_latency_us)
e.close()
"""


def test_first_probe_latency_is_that_of_the_next():
    """In a process of its own, where the probe's kernels have not run yet.  A round trip takes 15 to 30 us; to load one
    kernel's code takes 400, so a mean over ten turns with the load among them is 40 above."""
    r = subprocess.run([sys.executable, "-c", TWICE], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    first, second = (float(v) for v in r.stdout.split()[-2:])
    print(first, second, flush=True)
    assert first < second + 20.0
