"""Pinned staging memory between a Net and its callers (dabnn_amd/host/staging.cpp), over a runtime in host memory with two devices."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_on_either_of_two_devices(tmp_path):
    program, host = str(tmp_path / "staging_test"), os.path.join(ROOT, "dabnn_amd", "host")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", program,
                    os.path.join(ROOT, "tests", "cpp", "staging_test.cpp"), os.path.join(host, "mat.cpp"), os.path.join(host, "staging.cpp")], check=True)
    run = subprocess.run([program], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr
