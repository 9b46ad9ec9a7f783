"""The raycast forms a sample's texture coordinate x / width + 1/2 from the exact
reciprocal of the width; tests/cpp/width_div_check.c checks on the CPU that this
is the coordinate of the correctly rounded quotient."""
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_texture_coordinate_matches_rounded_quotient():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "width_div_check")
        subprocess.check_call(["gcc", "-O2", "-ffp-contract=off", "-o", exe,
                               os.path.join(HERE, "cpp", "width_div_check.c"), "-lm"])
        r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stdout
