"""The cut of marches and walks into chunks (miso_amd/csrc/split_rounds.hpp),
on the CPU by tests/cpp/test_split_rounds.cpp: the choice of a scan of every
count, at a cost that no launch notices.  It runs at every launch; scanning
every count took 140 us for a strip of 32790 rows and 440 for 100000."""
import ctypes
import os

import pytest

LIB = os.path.join(os.path.dirname(__file__), "cpp", "_build", "libsplit_rounds_check.so")
pytestmark = pytest.mark.skipif(not os.path.exists(LIB),
                                reason="tests/cpp not built (run __graft_entry__.build())")


def test_choice_is_that_of_a_full_scan():
    lib = ctypes.CDLL(LIB)
    msg, calls = ctypes.create_string_buffer(512), ctypes.c_int(0)
    rc = lib.split_rounds_check(msg, 512, ctypes.byref(calls))
    assert rc == 0, msg.value.decode()
    assert calls.value > 50000, calls.value


@pytest.mark.parametrize("n,per_chunk,slots", [(256, 1, 256), (32790, 1, 256), (100000, 1, 768),
                                               (16384, 61, 768), (100000, 4000, 256)])
def test_a_call_costs_far_less_than_a_launch(n, per_chunk, slots):
    lib = ctypes.CDLL(LIB)
    lib.split_rounds_time.restype = ctypes.c_double
    lib.split_rounds_time.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_int, ctypes.c_long]
    us = lib.split_rounds_time(n, per_chunk, 256, slots)
    assert us < 25.0, us


@pytest.mark.parametrize("ni,most,f64,want", [
    (1, 256, 1, 16), (8, 256, 1, 16), (8, 256, 0, 16), (8, 4, 1, 4), (9, 256, 1, 256),
    (64, 256, 1, 256), (65, 256, 1, 128), (72, 256, 1, 128), (72, 64, 1, 64), (72, 256, 0, 256),
    (73, 256, 1, 256), (512, 4096, 1, 4096)])
def test_narrow_rows_walk_short(ni, most, f64, want):
    """A last segment of at most eight cells: 72 x 512 x 512's z sweep in FP64
    takes 2220 us in walks of 256 planes and 958 in walks of 128."""
    assert ctypes.CDLL(LIB).walk_limit_of(ni, most, f64) == want


@pytest.mark.parametrize("nj,nseg,npl,nparts", [(128, 3, 130, 11), (96, 2, 98, 8), (64, 2, 66, 4),
                                                (300, 1, 92, 6)])
def test_slabs_of_the_xy_walk_fill_the_chip(nj, nseg, npl, nparts):
    """A slab of the overlapped walks has a few planes: the whole walk's cut
    would make 14 to 42 blocks of it, for 256 CUs."""
    lib, out = ctypes.CDLL(LIB), (ctypes.c_int * 2)()
    lib.split_xy_of(nj, nseg, npl, nparts, 64, out)
    chunk, n = out
    assert chunk * n >= nj and (n - 1) * chunk < nj
    waves = nseg * nparts
    assert (waves * n + 3) // 4 >= 128 or chunk == 1
    # slabs of a large box keep the whole walk's cut
    lib.split_xy_of(512, 9, 514, 32, 64, out)
    whole = tuple(out)
    lib.split_xy_of(512, 9, 514, 0, 64, out)
    assert tuple(out) == whole
