"""bench.py contract on the CPU: more than one GPU is refused with a message."""
import os
import subprocess
import sys

from conftest import ROOT


def test_multi_gpu_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "one GPU" in r.stderr


def test_fill_traffic_is_a_curves_share_per_launch():
    """The roofline's bytes per launch are the measured bytes of one curve's
    fill launches over their number."""
    import bench
    one = bench.measured_traffic(1)
    assert one > 1e8
    assert bench.measured_traffic(3.4) == one / 3.4
