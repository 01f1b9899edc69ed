"""The reactive path's counters (mcell_amd/csrc/device/header.h), host build:
the reactions of a call and their log rows are 64-bit numbers (a call may
cover any number of iterations), the output slots end at the capacity."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("header") / "libheader.so"
    subprocess.check_call([hipcc, "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                           os.path.join(HERE, "header_shim.cpp"), "-o", str(out)])
    lib = ctypes.CDLL(str(out))
    lib.book_phases.restype = ctypes.c_uint64
    lib.book_slots.restype = ctypes.c_uint32
    return lib


@pytest.mark.parametrize("before", [0, 2 ** 32 - 1500, 2 ** 32 - 1, 2 ** 32, 2 ** 40 + 3])
def test_reactions_of_a_call_past_32_bits(shim, before):
    n = np.array([1000, 1, 700, 2 ** 31], np.uint32)
    rows = np.zeros((len(n), 2), np.uint64)
    total = shim.book_phases(ctypes.c_uint64(before), ctypes.c_uint64(len(n)), ctypes.c_void_p(n.ctypes.data),
                             ctypes.c_void_p(rows.ctypes.data))
    base = before
    for k, (first, last) in zip(n.tolist(), rows.tolist()):
        assert (first, last) == (base, base + k - 1)
        base += k
    assert total == base


@pytest.mark.parametrize("used,total,capacity", [(0, 0, 10), (7, 3, 10), (7, 4, 10), (2 ** 32 - 2, 2 ** 31, 2 ** 32 - 1)])
def test_slots_end_at_the_capacity(shim, used, total, capacity):
    first = ctypes.c_uint32()
    assert shim.book_slots(used, ctypes.c_uint32(total), ctypes.c_uint32(capacity),
                           ctypes.byref(first)) == min(used + total, capacity)
    assert first.value == used
