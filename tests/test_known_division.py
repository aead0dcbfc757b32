"""The kernels' division by a known value (two-part reciprocal and one exact
residual) gives the IEEE quotient, bit for bit: compiled for the host, where
the hardware's division is the oracle."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_known_division_is_the_ieee_quotient(tmp_path):
    exe = str(tmp_path / "known_division")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "native", "known_division.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    bad, n = (int(v) for v in out.stdout.split())
    assert n > 5_000_000 and bad == 0, out.stdout
