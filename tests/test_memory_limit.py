"""Plans at the limit of device memory, with a stand-in for the HIP layer (host only, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plans_at_the_memory_limit():
    prog = os.path.join(ROOT, "tests", "c", "_build", "test_memory_limit")
    out = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout
