"""The radix steps with lazy reduction (ntt_amd/csrc/radix.h) on the host: slots at the ends of their ranges in every sign
pattern, twiddles at theirs, for every group size, with and without trivial twiddles and wide inputs and outputs.  Every
operand of a product or reduction stays within 4p (mul_shoup's and reduce's range), outputs within what the next step
takes, and every output is exact modulo p."""
import ctypes as C
import os
import subprocess
from fractions import Fraction

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "radix_host.cpp")
SO = os.path.join(HERE, "native", "radix_host.so")
CS = os.path.join(HERE, "..", "ntt_amd", "csrc")


@pytest.fixture(scope="module")
def R():
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(os.path.getmtime(f) for f in (
            SRC, os.path.join(CS, "radix.h"), os.path.join(CS, "arith.h"))):
        tmp = "%s.%d.tmp" % (SO, os.getpid())
        subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-fPIC", "-shared",
                        "-o", tmp, SRC], check=True)
        os.replace(tmp, SO)
    L = C.CDLL(SO)
    L.r_radix.argtypes = [C.c_int] * 6 + [C.c_uint64, C.c_uint64, C.POINTER(C.c_double)]; L.r_radix.restype = C.c_int
    L.r_mask.argtypes = [C.c_int] * 3; L.r_mask.restype = C.c_uint32
    L.r_prime.argtypes = [C.c_int]; L.r_prime.restype = C.c_uint64
    return L


def radix(R, logr, inv, triv, wide_in, wide_out, prime):
    most = (C.c_double * 3)()
    bad = R.r_radix(logr, inv, triv, wide_in, wide_out, prime, 0, max(1 << (1 << logr), 4096), most)
    return bad, [int(x) for x in most]


@pytest.mark.parametrize("prime", [0, 3])
@pytest.mark.parametrize("triv", [0, 1])
@pytest.mark.parametrize("logr", [1, 2, 3, 4])
def test_dif(R, logr, triv, prime):
    """inputs within p; outputs within p, plus the 1 by which each of two reduced terms may pass p / 2"""
    p = R.r_prime(prime)
    bad, (mul, red, out) = radix(R, logr, 0, triv, 0, 0, prime)
    assert not bad and mul <= 4 * p and red <= 4 * p and out <= p + 2


@pytest.mark.parametrize("prime", [0, 3])
@pytest.mark.parametrize("wide_in", [0, 1])
@pytest.mark.parametrize("wide_out", [0, 1])
@pytest.mark.parametrize("triv", [0, 1])
@pytest.mark.parametrize("logr", [1, 2, 3, 4])
def test_dit(R, logr, triv, wide_in, wide_out, prime):
    """inputs within p or 4p; outputs within 4p, or reduced"""
    p = R.r_prime(prime)
    bad, (mul, red, out) = radix(R, logr, 1, triv, wide_in, wide_out, prime)
    assert not bad and mul <= 4 * p and red <= 4 * p and out <= (4 * p if wide_out else p // 2 + 1)


@pytest.mark.parametrize("triv", [0, 1])
@pytest.mark.parametrize("logr", [1, 2, 3, 4])
def test_dif_mask_bounds(R, logr, triv):
    """the reductions that DifRed names keep every slot's bound (in exact fractions of p, a reduced value counted p / 2 and
    2^-40 more): within 4 at every product and reduction, within 1 and 2^-30 at the end"""
    n = 1 << logr
    half = Fraction(1, 2) + Fraction(1, 2 ** 40)
    b = [Fraction(1)] * n
    for lev in range(logr):
        h, mask = n >> (lev + 1), R.r_mask(logr, triv, lev)
        for jj in range(h):
            for j in range(jj, n, 2 * h):
                s = b[j] + b[j + h]
                assert s <= 4
                b[j] = half if (mask >> j) & 1 else s
                if triv and jj == 0:
                    b[j + h] = half if (mask >> (j + h)) & 1 else s
                else:
                    b[j + h] = Fraction(1, 2) + s / 16
    assert max(b) <= 1 + Fraction(1, 2 ** 30)
