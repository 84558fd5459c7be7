"""The stencil lanes' LDS addresses (csrc/stencil_lanes.hpp) on the host: no
lane reads past its plane, lanes without a point of their own included."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lds_reads_stay_in_the_plane(tmp_path):
    exe = str(tmp_path / "stencil_lanes")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "lynx_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "stencil_lanes.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
