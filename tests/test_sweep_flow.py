"""The flow control between the waves of a triangular sweep, walked on the host: tests/cpp/sweep_flow.cpp runs the
waves in every order against the rules the kernel uses (nlf_sweep_flow.hpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_wave_overwrites_what_another_still_reads(tmp_path):
    exe = str(tmp_path / "sweep_flow")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{ROOT}/nonlocal_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "sweep_flow.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout
