"""Device-to-host copies (ipglasma_amd/csrc/copy_out.hpp) on a stand-in for the
HIP runtime: whatever way a copy takes, it comes after the work queued on its
own context's stream, waits for no other context's, and leaves nothing queued."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host", "copy_out_host.cpp")
OUT = os.path.join(HERE, "_build", "libcopy_out_host.so")
PAGEABLE, PINNED, DEVICE, MANAGED = range(4)
KEYS = ("status", "right", "drained_other", "null_copies", "direct", "slots", "error", "alive")


@pytest.fixture(scope="module")
def lib():
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fPIC", "-shared", "-pthread", "-o", OUT, SRC], check=True,
                   capture_output=True)
    L = C.CDLL(OUT)
    L.copy_out_case.argtypes = [C.c_longlong, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_longlong)]
    L.copy_out_slot.restype = C.c_longlong
    return L


def case(lib, n, kind=PAGEABLE, busy=0, fail=0):
    out = (C.c_longlong * 8)()
    lib.copy_out_case(n, kind, busy, fail, out)
    return dict(zip(KEYS, out))


def sizes(lib):
    s = lib.copy_out_slot()
    # one value, below the slots' threshold, at it, short last chunks, more chunks than slots
    return [8, 2 * s - 8, 2 * s, 2 * s + 8, 3 * s + 1, 19 * s + 12345]


@pytest.mark.parametrize("k", range(6))
@pytest.mark.parametrize("busy,fail", [(0, 0), (1, 0), (0, 1), (0, 3)])
def test_pageable_copy_waits_for_its_own_stream_only(lib, k, busy, fail):
    n = sizes(lib)[k]
    r = case(lib, n, busy=busy, fail=fail)
    assert r["status"] == 0 and r["right"] == 1 and r["error"] == 0, r
    assert r["drained_other"] == 0 and r["null_copies"] == 0, r
    assert r["direct"] + r["slots"] == n and r["alive"] == 0, r
    if busy or fail == 1:  # no slots: one plain copy
        assert r["direct"] == n, r


def test_failed_slot_copy_is_reported(lib):
    r = case(lib, 19 * lib.copy_out_slot(), fail=2)
    assert r["status"] == 1 and r["alive"] == 0, r


@pytest.mark.parametrize("k", range(6))
@pytest.mark.parametrize("kind", [PINNED, DEVICE, MANAGED])
def test_destination_the_device_reaches_takes_one_copy(lib, k, kind):
    """not the slots, whose memcpy is slower than the DMA into pinned memory and
    wrong for device memory"""
    n = sizes(lib)[k]
    r = case(lib, n, kind=kind)
    assert r["status"] == 0 and r["right"] == 1 and r["error"] == 0, r
    assert r["direct"] == n and r["slots"] == 0, r
    assert r["drained_other"] == 0 and r["null_copies"] == 0, r
