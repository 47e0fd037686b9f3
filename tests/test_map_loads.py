"""The field map's cell records are read with global loads in every kernel of
the built library.  A flat load, which the compiler takes where it cannot
tell global memory from LDS, waits for the wavefront's LDS accesses too."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

from acts_amd.build import LIB_PATH

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def _wide_flat_loads(code_object):
    """{kernel: number of flat loads wider than one word}, and the kernels."""
    out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code_object],
                         capture_output=True, text=True, check=True).stdout
    found, kernels, name = {}, [], None
    for line in out.splitlines():
        head = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if head:
            name = head.group(1)
            kernels.append(name)
        elif "flat_load_dwordx" in line:
            found[name] = found.get(name, 0) + 1
    return found, kernels


def test_no_wide_flat_loads(tmp_path):
    lib = shutil.copy(LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], capture_output=True, check=True,
                   cwd=tmp_path)
    objects = [str(tmp_path / f) for f in os.listdir(tmp_path) if "gfx950" in f]
    with ThreadPoolExecutor(4) as pool:
        found = list(pool.map(_wide_flat_loads, objects))
    assert any("fitForwardKernel" in k for _, kernels in found for k in kernels)
    assert {k: n for f, _ in found for k, n in f.items()} == {}
