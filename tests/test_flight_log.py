"""The flight draws' logarithm against the long double one."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_flight_log_error(tmp_path):
    """Every interval's ends, the neighbourhood of 0 and 1 and 6e5 draws: the
    rounding of the last addition, 0.5 ulp, and up to 2^-8 relative of the
    terms that are added to the leading one with an error of 0.5 ulp of their
    own, a dozen of them at most: below 0.55 ulp. log 1 is 0."""
    exe = str(tmp_path / "flight_log_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-D__device__=", "-D__host__=", "-I",
                    os.path.join(ROOT, "bte-barna_amd", "csrc"), os.path.join(ROOT, "tests", "flight_log_check.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe, "200000"], check=True, capture_output=True, text=True).stdout.split()
    assert float(out[0]) < 0.55, out
