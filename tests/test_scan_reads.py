"""The scan's reads of the segment totals on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reads_stay_in_the_totals(tmp_path):
    """No thread reads past the first padding entry, behind which other
    workgroups may be writing (tests/golden/scan_read_check.cpp)."""
    exe = tmp_path / "scan_read_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "framework_amd", "csrc"),
                    os.path.join(ROOT, "tests", "golden", "scan_read_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120).stdout
    assert out.strip() == "OK", out
