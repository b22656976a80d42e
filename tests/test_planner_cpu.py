"""The planner's choices without a device (tests/cpp/planner_check.cpp): untuned plans take fast
splits, real ones with the price of their split, and the pruned search finds the best."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_planner_choices():
    exe = os.path.join(HERE, "cpp", "planner_check")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
