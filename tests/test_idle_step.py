"""An electron that stands at the synchronization time already (a collision or an
ejection exactly there) leaves the flight step bit for bit as it entered, with no
field gain: the device's step function compiled for the host, over all field cases
and both forms."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_step_at_the_synchronization_time_changes_nothing(tmp_path):
    exe = str(tmp_path / "idle_step")
    native = os.path.join(ROOT, "tests", "native")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I" + os.path.join(native, "host"),
                    os.path.join(native, "idle_step.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    bad, n = (int(v) for v in out.stdout.splitlines()[-1].split())
    assert n == 280_000 and bad == 0, out.stdout
