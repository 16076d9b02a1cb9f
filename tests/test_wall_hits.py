"""The counters of a wall whose step and emission hits may cancel."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_wave_takes_the_same_hits(tmp_path):
    exe = str(tmp_path / "wall_hits_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__device__=", "-D__host__=", "-I",
                    os.path.join(ROOT, "bte-barna_amd", "csrc"), os.path.join(ROOT, "tests", "wall_hits_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
