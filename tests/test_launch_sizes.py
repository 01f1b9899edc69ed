"""Launch sizes of the reactive path (mcell_amd/csrc/launch_sizes.h), host
build: no kernel is left to a few workgroups where its work needs a grid, and
none gets workgroups it has no use for."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
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
    for f in (lib.scatter, lib.append, lib.room):
        f.restype = ctypes.c_uint32
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


def test_first_rounds_are_sized_by_the_same_phase(shim):
    """Iterations whose phases need reruns, the last of which brings nothing:
    from the second iteration on every phase's first round is expected as it
    was, whatever the rounds between, and a rerun as its list."""
    it = [  # phase, round, form, movers, proposals, deferred
        (0, 0, 1, 10 ** 6, 50000, 9000), (0, 1, 1, 4000, 1500, 10), (0, 2, 1, 100, 0, 0),
        (1, 0, 1, 150000, 30000, 7000), (1, 1, 1, 5000, 0, 0),
        (2, 0, 1, 90000, 800, 0), (2, 1, 1, 20, 0, 0),
        (9, 0, 1, 500, 40, 3), (10, 0, 1, 400, 30, 2)]
    rounds = np.array(it * 3, np.uint32)
    out = np.zeros((len(rounds), 2), np.uint32)
    shim.rounds(ctypes.c_uint64(len(rounds)), ctypes.c_void_p(rounds.ctypes.data), ctypes.c_void_p(out.ctypes.data))
    for i, (phase, rnd, _, movers, props, deferred) in enumerate(rounds.tolist()):
        if rnd:
            assert out[i].tolist() == [movers, movers]
        elif i < len(it):
            # nothing known yet: all movers (phases past the eighth share a slot)
            assert phase == 10 and out[i].tolist() == [40, 3] or out[i].tolist() == [movers, movers]
        elif phase < 9:
            assert out[i].tolist() == [props, deferred]


def test_forms_are_told_apart(shim):
    rounds = np.array([(0, 0, 1, 1000, 10, 0), (0, 0, 2, 1000, 10, 700), (0, 0, 1, 1000, 10, 0), (0, 0, 2, 1000, 0, 0)],
                      np.uint32)
    out = np.zeros((4, 2), np.uint32)
    shim.rounds(ctypes.c_uint64(4), ctypes.c_void_p(rounds.ctypes.data), ctypes.c_void_p(out.ctypes.data))
    assert out.tolist() == [[1000, 1000], [1000, 1000], [10, 0], [10, 700]]


@pytest.mark.parametrize("expected,bound,room", [(0, 10, 10), (0, 1000, 64), (100, 1000, 264),
                                                 (2 ** 31, 2 ** 32 - 1, 2 ** 32 - 1), (2 ** 32 - 1, 5, 5)])
def test_room_for_twice_the_expected(shim, expected, bound, room):
    assert shim.room(ctypes.c_uint32(expected), ctypes.c_uint32(bound)) == room
