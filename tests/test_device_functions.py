"""Device functions of the built library that the compiler left out of line.

A function that can see a pointer to LDS or private memory has to be inlined (see nuts_device.h); the
ones named here take scalars and global-memory pointers only."""
import os
import re
import shutil
import subprocess

import pytest

from cmdstan_amd import LIB_PATH

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
OUT_OF_LINE = {"stream_normal", "dense_matvec", "dense_matvec2", "dense_inverse"}


def device_functions(tmp_path):
    """Names of the functions of every code object that are no kernels (a kernel has a descriptor NAME.kd)."""
    lib = str(tmp_path / "lib.so")
    shutil.copy(LIB_PATH, lib)
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], check=True, cwd=tmp_path,
                   capture_output=True)
    objs = [str(p) for p in tmp_path.iterdir() if p.name.startswith("lib.so.") and "gfx950" in p.name]
    names, kernels = set(), 0
    for o in objs:
        t = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "-sW", o], check=True, capture_output=True, text=True)
        sym = [(f[3], f[7]) for f in (line.split() for line in t.stdout.splitlines()) if len(f) >= 8]
        kd = {n[:-3] for _, n in sym if n.endswith(".kd")}
        kernels += len(kd)
        names |= {n for kind, n in sym if kind == "FUNC" and n not in kd}
    return names, kernels


@pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-objdump")), reason="no ROCm LLVM tools")
def test_out_of_line_device_functions(tmp_path):
    names, kernels = device_functions(tmp_path)
    assert kernels > 100
    found = set()
    for n in names:
        m = re.match(r"_ZN7nutsgpuL?(\d+)(\w+)", n)
        found.add(m[2][:int(m[1])] if m else n)
    assert found <= OUT_OF_LINE, found - OUT_OF_LINE
