"""The exponential of a pre-scaled argument (mdt_exp_t in
md_tian2_amd/csrc/mdt_math.h), compiled for the host, within its bound against
libm over the range that the pair terms use and to the ends of its own."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_mdt_exp_t_within_its_bound():
    src = os.path.join(ROOT, "tests", "native", "exp_t_check.c")
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "exp_t_check")
        subprocess.run(["gcc", "-O2", "-o", exe, src, "-lm"], check=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert float(out[0]) <= 1.0, out
