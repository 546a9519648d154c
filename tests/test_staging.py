"""Pinned staging memory between a Net and its callers (dabnn_amd/host/staging.cpp), over a runtime in host memory with two devices."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("events", [16, 4, 2])
def test_copies_on_either_of_two_devices(tmp_path, events):
    """With fewer events as well, so that transfers that overwrite each other's pinned memory share one."""
    program, host = str(tmp_path / "staging_test"), os.path.join(ROOT, "dabnn_amd", "host")
    for name in ("staging.h", "staging.cpp", "mat.h", "mat.cpp"):
        text = open(os.path.join(host, name)).read()
        (tmp_path / name).write_text(text.replace("kEvents = 16", "kEvents = %d" % events))
    test = open(os.path.join(ROOT, "tests", "cpp", "staging_test.cpp")).read().replace("../../dabnn_amd/host/", "")
    (tmp_path / "staging_test.cpp").write_text(test)
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", program] +
                   [str(tmp_path / name) for name in ("staging_test.cpp", "mat.cpp", "staging.cpp")], check=True)
    run = subprocess.run([program], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr
