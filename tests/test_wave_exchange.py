"""A wave's exchanges through LDS (mdmc_wave.h) on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lanes_in_any_order_between_the_points(tmp_path):
    """Lanes run one after the other between the order points, in random
    sequences: every value arrives (tests/golden/wave_exchange_check.cpp)."""
    exe = tmp_path / "wave_exchange_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "framework_amd", "csrc"),
                    os.path.join(ROOT, "tests", "golden", "wave_exchange_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout
    assert out.strip() == "OK", out
