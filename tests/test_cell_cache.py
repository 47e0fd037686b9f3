"""The lane's copy of its last field-map cell (CellCache in
acts_amd/csrc/kf_device.hpp) serves every cell-major map: the ones whose axes
multiply by reciprocals and the ones whose axes divide, in both precisions.
The lookups are compiled for the host (tests/cpp/cell_cache_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lookups_keep_their_cell(tmp_path):
    exe = str(tmp_path / "cell_cache_check")
    res = subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-w",
                          "-I", os.path.join(HERE, "cpp", "hip_stub"), "-o", exe,
                          os.path.join(HERE, "cpp", "cell_cache_check.cpp")],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout + res.stderr
