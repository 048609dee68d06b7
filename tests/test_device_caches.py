"""The library's process-wide caches follow the current device (CPU; a fake HIP)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("caches") / "libdevicecaches.so")
    src = os.path.join(ROOT, "tests", "hostmath", "device_caches.cpp")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", "-Wl,-Bsymbolic",
                    "-fno-gnu-unique", "-I/opt/rocm/include", "-o", so, src], check=True)
    return C.CDLL(so)


def test_constants_stay_on_their_device(lib):
    """Grid tables, tau sets and flow constants are shared by everything on one device and
    by nothing on another one, also while an object on the first keeps them."""
    assert lib.shared_between(0, 0) == 3
    assert lib.shared_between(0, 1) == 0
    assert lib.shared_between(1, 1) == 3


def test_lds_limit_is_raised_on_every_device(lib):
    """A kernel above 64 KB of LDS is opted in once on each device that launches it."""
    assert lib.raises(3, C.c_long(64 * 1024)) == 0
    assert lib.raises(3, C.c_long(100 * 1024)) == 3
    assert lib.raises(3, C.c_long(100 * 1024)) == 0
