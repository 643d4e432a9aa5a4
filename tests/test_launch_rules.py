"""The launch rules of the lvl1 rotations (launch_rules.hpp), compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launch_rules():
    exe = os.path.join(ROOT, "tests", "cpp", "test_launch_rules.bin")
    assert os.path.exists(exe), "build first: python cufhe_amd/build.py"
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.startswith("ok:"), p.stdout + p.stderr
