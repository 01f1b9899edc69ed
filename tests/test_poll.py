"""The wait for the host's copy of the counters (mcell_amd/csrc/poll.h), host
build: it spins for a short while only, then gives its core away between two
looks, asks the runtime seldom, and ends when nothing more can come."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
NEVER = 2 ** 64 - 1


@pytest.fixture(scope="module")
def poll(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    out = tmp_path_factory.mktemp("poll") / "libpoll.so"
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "poll_shim.cpp"),
                           "-o", str(out)])
    lib = ctypes.CDLL(str(out))

    def call(ready_at, rest_at):
        c = np.zeros(4, np.uint64)
        there = lib.poll(ctypes.c_uint64(ready_at), ctypes.c_uint64(rest_at), ctypes.c_void_p(c.ctypes.data))
        return bool(there), *c.tolist()

    return call


@pytest.mark.parametrize("ready_at", [0, 1, 999, 1000, 1001, 50000, 10 ** 6])
def test_yields_after_a_short_spin(poll, ready_at):
    there, looks, pauses, yields, queries = poll(ready_at, NEVER)
    assert there and looks == ready_at + 1
    assert pauses == min(ready_at, 1000) and pauses + yields == ready_at
    assert ready_at // 40000 <= queries <= ready_at // 10000


@pytest.mark.parametrize("rest_at", [0, 3])
def test_ends_when_nothing_more_can_come(poll, rest_at):
    there, looks, _, _, queries = poll(NEVER, rest_at)
    assert not there and queries == rest_at + 1
    # the word that came while the runtime was asked is still seen
    assert poll(looks - 1, rest_at)[0]
