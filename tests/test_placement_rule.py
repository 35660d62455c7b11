"""Runs of tiles placed side by side on one XCD: counted in slices, so that a
launch of few but large tiles is not left to the memory rate of one or two
XCDs (tests/cpp/xcd_run_check.cpp).  And the XCDs that concurrent contexts start on
(tests/cpp/xcd_start_check.cpp)."""
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


def test_concurrent_contexts_start_apart(tmp_path):
    exe, lib = str(tmp_path / "xcd_start_check"), os.path.join(HERE, "..", "mprgp_amd")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "cpp", "xcd_start_check.cpp"),
                    "-L", lib, "-lmprgp_amd", "-Wl,-rpath," + os.path.abspath(lib), "-Wl,--allow-shlib-undefined",
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
