"""The torus rounding of the FP64 backends (double_to_torus, turns_to_torus32) and the
distance of the lvl1 products from the integers that they round to, compiled for the
host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_double_to_torus_matches_integer_rounding():
    exe = os.path.join(ROOT, "tests", "cpp", "test_torus_convert.bin")
    assert os.path.exists(exe), "build first: python cufhe_amd/build.py"
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.startswith("ok:"), p.stdout + p.stderr


def test_lvl1_products_are_near_their_integers():
    exe = os.path.join(ROOT, "tests", "cpp", "test_lvl1_rounding.bin")
    assert os.path.exists(exe), "build first: python cufhe_amd/build.py"
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and "ok:" in p.stdout, p.stdout + p.stderr
