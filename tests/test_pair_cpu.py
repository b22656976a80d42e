"""Lanes of the paired real-transform tiles stay inside the pass-twiddle tables (host walk)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_paired_lanes_index_inside_the_pass_tables():
    exe = os.path.join(HERE, "cpp", "pair_check")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
