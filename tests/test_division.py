"""The division sequence of the 2-D patches' geometry, over every significand
(tests/cpuemu/check_division.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_division_rounds_correctly(tmp_path):
    exe = str(tmp_path / "check_division")
    emu = os.path.join(HERE, "cpuemu")
    subprocess.run(["g++", "-std=c++20", "-O2", "-I" + emu, "-I" + os.path.join(HERE, "..", "specfempp_amd", "csrc"),
                    os.path.join(emu, "check_division.cpp"), "-o", exe, "-lpthread"], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
