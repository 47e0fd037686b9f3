"""The copies between a caller's arrays and the device through pinned memory
(acts_amd/csrc/kf_host_copy.hpp) where threads or memory run out or a copy
fails: a C entry point must return then, not end the process.  Compiled for the
host with a stand-in runtime (tests/cpp/host_copy_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_copies_without_threads_or_memory(tmp_path):
    exe = str(tmp_path / "host_copy_check")
    res = subprocess.run(["g++", "-O2", "-std=c++17", "-pthread",
                          "-I", os.path.join(HERE, "cpp", "hip_stub"), "-o", exe,
                          os.path.join(HERE, "cpp", "host_copy_check.cpp"), "-ldl"],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0 and res.stdout == "ok\n", (res.returncode, res.stdout, res.stderr)
