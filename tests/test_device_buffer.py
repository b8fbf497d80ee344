"""The growable device buffer after an allocation that failed: a call that
runs out of memory reports it, and the next call with a smaller grid must not
find the capacity of the buffer that was given up (its kernels would write to
a null pointer)."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("devbuf") / "devbuf_alloc.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                           "-I", os.path.join(rocm, "include"), "-o", so,
                           os.path.join(HERE, "helpers", "devbuf_alloc.cpp")])
    L = ctypes.CDLL(so)
    L.grow_fail_grow.argtypes = [ctypes.c_size_t] * 3
    return L


@pytest.mark.parametrize("first,more,after", [(1, 5000, 1), (1024, 1025, 1024), (3000, 1 << 20, 4096),
                                              (3000, 1 << 20, 1 << 20)])
def test_buffer_after_a_failed_allocation(lib, first, more, after):
    assert lib.grow_fail_grow(first, more, after) == 1
