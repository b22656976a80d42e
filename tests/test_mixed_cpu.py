"""The run-time mixed-radix tiles' shapes, walked on the CPU (tests/cpp/mixed_check.cpp): every
length with the factors 2, 3, 5 and 7 a tile takes, every mode, width and precision."""
import os
import subprocess

import pytest

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "mixed_check")


def test_every_tile_shape():
    if not os.path.exists(CHECK):
        pytest.skip("tests/cpp/mixed_check is not built (__graft_entry__.build())")
    r = subprocess.run([CHECK], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
