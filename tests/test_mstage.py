"""CNOT / SWAP / CZ stages folded into the passes as index maps and signs: the C program
compares them with the gates applied one by one (host only, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_index_maps_and_signs():
    prog = os.path.join(ROOT, "tests", "c", "_build", "test_mstage")
    out = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout
