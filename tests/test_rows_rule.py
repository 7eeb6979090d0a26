"""The rule for wide and unaligned rows (csrc/rows_wide.hpp), replayed on the CPU: no call it takes has a
grid that a launch would refuse."""
import os
import subprocess

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_rows_rule_stays_within_a_launch():
    subprocess.run(["make", "-C", NATIVE, "rows_rule_check"], check=True, capture_output=True)
    r = subprocess.run([os.path.join(NATIVE, "rows_rule_check")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
