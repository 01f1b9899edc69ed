"""Launch sizes of the reactive path (mcell_amd/csrc/launch_sizes.h), host
build: no kernel is left to a few workgroups where its work needs a grid, and
none gets workgroups it has no use for."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    out = tmp_path_factory.mktemp("launch") / "liblaunch.so"
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "launch_shim.cpp"),
                           "-o", str(out)])
    lib = ctypes.CDLL(str(out))
    lib.scatter.restype = lib.append.restype = ctypes.c_uint32
    return lib


@pytest.mark.parametrize("molecules", [0, 1, 200, 256, 257, 4000, 10 ** 6, 10 ** 8])
@pytest.mark.parametrize("bins", [1, 4096, 4097, 10 ** 5, 54 * 10 ** 6, 0xFFFFFFEF])
def test_scatter_clears_the_bins_with_enough_threads(shim, molecules, bins):
    wg = shim.scatter(ctypes.c_uint32(molecules), ctypes.c_uint32(bins))
    own = max(1, -(-molecules // 256))
    assert wg >= own
    assert wg >= 2048 or wg * 256 * 16 >= bins     # at most 16 bins a thread, or the whole chip
    assert wg == own or wg <= 2048 and (wg - 1) * 256 * 16 < bins  # no more than that takes


@pytest.mark.parametrize("entries", [1, 256, 16384, 16385, 10 ** 6, 0xFFFFFFFF])
def test_long_lists_are_copied_by_a_grid(shim, entries):
    wg = shim.append(ctypes.c_uint32(entries))
    if wg == 1:
        assert entries <= 16 * 1024  # sixteen turns of the lone workgroup of 1,024
    else:
        assert wg == 2048 or (wg - 1) * 256 < entries <= wg * 256
