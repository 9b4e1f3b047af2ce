"""Every LDS access of the standard scheme's kernels lies in the plane of its
level: the planes' geometry (csrc/std_planes.hpp) against the rows and columns
the kernels read and write, walked over all waves and lanes on the host."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lds_accesses_stay_in_their_planes(tmp_path):
    exe = str(tmp_path / "std_planes_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "std_planes_check.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
