"""CPU tier: every read of X in the Heff W pass lies inside its LDS, for every
operator size the apply takes (Q (64 + O) <= 8192)."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def wp(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("wpass") / "libwpass.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "wpass_harness.cpp"), "-o", out], check=True)
    L = C.CDLL(out)
    L.wpass_last_read.restype = L.wpass_size.restype = C.c_int64
    L.wpass_tiles.argtypes = [C.c_int64]
    L.wpass_taken.argtypes = [C.c_int64, C.c_int64]
    return L


def test_reads_stay_inside(wp):
    for Q in range(1, 127):
        top = 8192 // Q - 64
        for O in sorted({1, 2, 15, 16, 17, 31, 32, 33, 45, 48, 49, 64, 65, 80, 96, 112, 128, top}):
            if O <= top and wp.wpass_size(Q, O, 4) * 8 <= 65536:
                nt = wp.wpass_tiles(O)
                assert wp.wpass_last_read(Q, O, nt) < wp.wpass_size(Q, O, nt), (Q, O)


def test_slices(wp):
    """the operators taken are those with Q (64 + O) <= 8192, and each is cut
    into launches whose X fits in 64 KB"""
    for Q in list(range(1, 140)) + [512, 600, 8192]:
        for O in sorted({1, 15, 16, 17, 33, 45, 80, 137, 340, 2000, 8128, 8192 // Q - 64, 8192 // Q - 63}):
            if O < 1:
                continue
            assert wp.wpass_taken(Q, O) == (Q * 64 + Q * O <= 8192)
            nt = wp.wpass_tiles(O)
            os_ = wp.wpass_slice(Q, O, nt)          # returns for any Q
            assert 1 <= os_ <= O
            if wp.wpass_taken(Q, O):
                assert wp.wpass_size(Q, os_, nt) * 8 <= 65536
