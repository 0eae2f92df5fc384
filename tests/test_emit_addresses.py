"""The emit's address arithmetic (mdmc_tilemap.h) on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_division_and_lane_offsets(tmp_path):
    """Division by multiplication is exact, and lane offsets within emit_span
    fit in 32 bits (tests/golden/emit_address_check.cpp)."""
    exe = tmp_path / "emit_address_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "framework_amd", "csrc"),
                    os.path.join(ROOT, "tests", "golden", "emit_address_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout
    assert out.strip() == "OK", out
