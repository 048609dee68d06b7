"""Register use of the built kernels, read from the library's own code objects."""
import os
import re
import shutil
import subprocess

import pytest

import channelflow_amd as cfa

LLVM = "/opt/rocm/llvm/bin"


def test_tau_solve_leaves_two_waves_per_simd(tmp_path):
    """The tau solve's instances of 32- and 64-lane segments (Ny from 193 on) take at most
    half of a SIMD's 512 registers and no scratch: with more, a block of 4 modes has its
    compute unit to itself and nothing runs while its rows are loaded."""
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("llvm-objdump not installed")
    lib = shutil.copy(os.path.join(os.path.dirname(cfa.__file__), "libcfgpu.so"), tmp_path)
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", os.path.basename(lib)], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    found = {}
    for f in os.listdir(tmp_path):
        if "amdgcn" not in f:
            continue
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", f], cwd=tmp_path, check=True,
                               capture_output=True, text=True).stdout
        for entry in notes.split(".agpr_count")[1:]:
            m = re.search(r"\.name:\s+\S*k_tau_solve_(?:wave|tall)ILi(\d+)ELi(\d+)E", entry)
            if m and int(m.group(2)) > 16:
                found[m.groups()] = [int(re.search(r"\.%s:\s+(\d+)" % k, entry).group(1))
                                     for k in ("vgpr_count", "private_segment_fixed_size")]
    print(found, flush=True)
    assert found and all(v <= 256 and s == 0 for v, s in found.values()), found
