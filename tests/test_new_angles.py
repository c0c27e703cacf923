"""New angles rebuild only a plan's matrices: the C program compares every descriptor with a
plan built at those angles (host only, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_new_angles_equal_a_fresh_build():
    prog = os.path.join(ROOT, "tests", "c", "_build", "test_new_angles")
    out = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout
