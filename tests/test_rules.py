"""The kernels' index arithmetic and launch rules on the CPU (native/rules_drive,
which names the first value that is out of place)."""
import os
import subprocess

DRIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "rules_drive")


def test_rules_hold():
    r = subprocess.run([DRIVE], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
