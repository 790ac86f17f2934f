"""The dispatch rules that count workgroups against the device's CUs (ntt_amd/csrc/segrule.h), built for the host: on a
partition of the device with a fraction of the CUs, that fraction of the work takes the same path and the same split."""
import ctypes as C
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "segrule_host.cpp")
SO = os.path.join(HERE, "native", "segrule_host.so")
HDR = os.path.join(HERE, "..", "ntt_amd", "csrc", "segrule.h")


@pytest.fixture(scope="module")
def R():
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(os.path.getmtime(SRC), os.path.getmtime(HDR)):
        tmp = "%s.%d.tmp" % (SO, os.getpid())
        subprocess.run(["g++", "-O2", "-Wall", "-Werror", "-fPIC", "-shared", "-o", tmp, SRC], check=True)
        os.replace(tmp, SO)
    L = C.CDLL(SO)
    u64p = C.POINTER(C.c_uint64)
    L.t_seg_launch_us.argtypes = [C.c_uint64, C.c_uint32, C.c_uint64, C.c_int]; L.t_seg_launch_us.restype = C.c_double
    L.t_seg_choose.argtypes = [C.c_uint64, C.c_uint64, C.c_double, C.c_int, C.c_int]; L.t_seg_choose.restype = C.c_uint32
    L.t_seg_batch_per.argtypes = [u64p, u64p, C.c_size_t, C.c_int]; L.t_seg_batch_per.restype = C.c_uint32
    L.t_small_few.argtypes = [C.c_uint64, C.c_int, C.c_int]; L.t_small_few.restype = C.c_int
    return L


@pytest.mark.parametrize("ncu", [32, 64, 128, 256])
def test_rounds(R, ncu):
    """a launch takes as many rounds as its workgroups fill the CUs"""
    for S in (512, 2048, 4032):
        one = R.t_seg_launch_us(1, 1, S, ncu)
        assert R.t_seg_launch_us(ncu, 1, S, ncu) == one
        assert R.t_seg_launch_us(ncu + 1, 1, S, ncu) == 2 * one
        assert R.t_seg_launch_us(4 * ncu, 1, S, ncu) == 4 * one
        assert R.t_seg_launch_us(6 * ncu, 1, S, ncu) == 6.5 * one


@pytest.mark.parametrize("ncu", [32, 64, 128])
def test_share_of_the_device(R, ncu):
    rnd = random.Random(ncu)
    for _ in range(300):
        S = 64 * rnd.randint(8, 63)
        segs = 840 * 256 // ncu * rnd.randint(1, 60)             # whole workgroups on both, at 1 to 8 segments each
        most = rnd.uniform(30, 3000)
        assert R.t_seg_choose(segs, S, most, 256, 0) == R.t_seg_choose(segs * ncu // 256, S, most, ncu, 0)
        kinds = [(840 * rnd.randint(1, 3), 64 * rnd.randint(8, 63)) for _ in range(rnd.randint(1, 5))]
        arr = lambda v: (C.c_uint64 * len(v))(*v)
        many = kinds * (256 // ncu)
        assert R.t_seg_batch_per(arr([k[0] for k in many]), arr([k[1] for k in many]), len(many), 256) == \
            R.t_seg_batch_per(arr([k[0] for k in kinds]), arr([k[1] for k in kinds]), len(kinds), ncu)


def test_few(R):
    for logn in range(7, 13):
        for ncu in (32, 256):
            line = (ncu << 11) >> logn
            assert R.t_small_few(line, logn, ncu) and not R.t_small_few(line + 1, logn, ncu)


def test_forced(R):
    """a forced product takes segments whatever the other path's time"""
    assert R.t_seg_choose(7, 1024, 0.0, 256, 0) == 0
    assert R.t_seg_choose(7, 1024, 0.0, 256, 1) >= 1
