"""CPU check of the workspaces' growth rules (scratch.h, compiled by g++ over a counted heap): memory
that is short refuses nothing the smallest form fits, and a buffer only moves for a call that needs
more than every one before it."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KEPT, MOVED, FAILED = range(3)


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("scratch") / "libscratch_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", out,
                    os.path.join(ROOT, "tests", "native", "scratch_host.cpp")], check=True)
    lib = ctypes.CDLL(out)
    z, i = ctypes.c_size_t, ctypes.c_int
    lib.scratch_host_reset.argtypes = [z]
    lib.scratch_host_set.argtypes = [z, i]
    lib.scratch_host_fit.argtypes = [i, z, z]
    lib.scratch_host_try_grow.argtypes = [i, z]
    for f in ("bytes", "used"):
        getattr(lib, "scratch_host_" + f).restype = z
    lib.scratch_host_ptr.restype = ctypes.c_void_p
    return lib


def test_no_call_after_a_larger_one_allocates(L):
    L.scratch_host_reset(1 << 40)
    # small calls want more than large ones: the address stays all the same
    assert L.scratch_host_fit(0, 500, 500) == MOVED
    p, n = L.scratch_host_ptr(0), L.scratch_host_allocs()
    for need, want in ((2, 8500), (10, 4600), (500, 9000), (1, 10**9)):
        assert L.scratch_host_fit(0, need, want) == KEPT
    assert L.scratch_host_ptr(0) == p and L.scratch_host_allocs() == n and L.scratch_host_idles() == 0
    # a larger one takes what it wants, after the device is idle
    assert L.scratch_host_fit(0, 501, 9000) == MOVED
    assert L.scratch_host_bytes(0) == 9000 and L.scratch_host_used() == 9000 and L.scratch_host_idles() == 1
    # and later ones live in that as long as it holds their need
    assert L.scratch_host_fit(0, 8000, 8100) == KEPT and L.scratch_host_fit(0, 8200, 9500) == MOVED
    assert L.scratch_host_bytes(0) == 9500


def test_short_memory_falls_back_to_the_need(L):
    L.scratch_host_reset(1000)
    assert L.scratch_host_fit(0, 100, 5000) == MOVED and L.scratch_host_bytes(0) == 100
    assert L.scratch_host_fit(0, 900, 5000) == MOVED and L.scratch_host_bytes(0) == 900
    assert L.scratch_host_fit(0, 1001, 5000) == FAILED
    assert L.scratch_host_bytes(0) == 0 and L.scratch_host_used() == 0 and not L.scratch_host_ptr(0)
    assert L.scratch_host_fit(0, 900, 900) == MOVED


def test_spare_memory_keeps_what_it_has(L):
    L.scratch_host_reset(1000)
    L.scratch_host_try_grow(1, 400)
    p = L.scratch_host_ptr(1)
    L.scratch_host_try_grow(1, 700)   # beside the old one there is no room
    assert (L.scratch_host_bytes(1), L.scratch_host_ptr(1), L.scratch_host_used()) == (400, p, 400)
    L.scratch_host_try_grow(1, 300)
    assert L.scratch_host_bytes(1) == 400
    L.scratch_host_try_grow(1, 600)
    assert L.scratch_host_bytes(1) == 600 and L.scratch_host_used() == 600
    # given back when it is idle, and taken again
    L.scratch_host_set(1000, 1)
    assert L.scratch_host_give_back(1) == 0 and L.scratch_host_bytes(1) == 600
    L.scratch_host_try_grow(1, 1000)
    assert L.scratch_host_bytes(1) == 600 and L.scratch_host_used() == 600
    L.scratch_host_set(1000, 0)
    assert L.scratch_host_give_back(1) == 1 and L.scratch_host_used() == 0
    assert L.scratch_host_give_back(1) == 0
    L.scratch_host_try_grow(1, 900)
    assert L.scratch_host_bytes(1) == 900


def test_a_busy_device_keeps_the_buffer(L):
    L.scratch_host_reset(1 << 20)
    assert L.scratch_host_fit(0, 10, 10) == MOVED
    L.scratch_host_set(1 << 20, 1)
    p = L.scratch_host_ptr(0)
    assert L.scratch_host_fit(0, 20, 20) == FAILED
    assert L.scratch_host_ptr(0) == p and L.scratch_host_bytes(0) == 10
