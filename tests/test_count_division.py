"""The precision form's count update divides by the count + 1 from an exact reciprocal;
tests/cpp/count_div_check.c checks on the CPU that this is the correctly rounded
quotient for the divisors 130 to 256 (tests/test_exact_division.py has those below)."""
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_count_update_matches_rounded_quotient_above_129():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "count_div_check")
        subprocess.check_call(["gcc", "-O2", "-ffp-contract=off", "-o", exe,
                               os.path.join(HERE, "cpp", "count_div_check.c"), "-lm"])
        r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stdout
