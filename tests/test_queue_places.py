"""Where the tracks that may become loopers stand in the queue
(acts_amd/csrc/kf_queue.hpp), compiled for the host
(tests/cpp/queue_check.cpp): a permutation at every batch size and number of
such tracks, and spread over no more wavefronts than the batch size allows."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_places(tmp_path):
    exe = str(tmp_path / "queue_check")
    res = subprocess.run(["g++", "-O2", "-std=c++17", "-w",
                          "-I", os.path.join(HERE, "cpp", "hip_stub"), "-o", exe,
                          os.path.join(HERE, "cpp", "queue_check.cpp")],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout + res.stderr
