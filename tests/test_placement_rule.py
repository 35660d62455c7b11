"""Runs of tiles placed side by side on one XCD: counted in slices, so that a
launch of few but large tiles is not left to the memory rate of one or two
XCDs (tests/cpp/xcd_run_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_runs_hold_at_most_an_xcds_share_of_slices(tmp_path):
    exe = str(tmp_path / "xcd_run_check")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "cpp", "xcd_run_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
