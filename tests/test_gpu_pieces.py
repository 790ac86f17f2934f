"""Uneven products formed in pieces of the longer operand that share the shorter one's transform: the pieces' overlap at its
edges (a short operand of one limb, of half a transform), pieces that end with the operand and just after it, 2^k and 3 2^k
points, three and four primes, an added operand, the shorter operand first, cuts, and results beyond one launch's planes.
Against the oracle, limb for limb, or (long products) against the whole transform's result and the oracle's residues."""
import os

import numpy as np
import pytest

import oracle as O
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu
TOP = np.uint64(10 ** 18 - 1)


@pytest.fixture
def pieces(nttm):
    import torch

    def set_(points=None, par=None, **cfg):
        for k, v in (("NTTM_PIECES", points), ("NTTM_PAR_POINTS", par)):
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = str(v)
        torch.cuda.synchronize()
        nttm.shutdown()
        nttm.init(0, **cfg)
        return nttm
    yield set_
    set_()


# points of the pieces' transforms; the pieces hold (points - nb + 1) & ~31 limbs
@pytest.mark.parametrize("points,na,nb", [
    (1 << 13, 16384 * 2, 1),             # one-limb operand: no overlap; 4 pieces, whole ones
    (1 << 13, 8192 * 3 + 1, 2),          # the last piece one limb or a few
    (1 << 13, 30011, 2100),
    (1 << 13, 20000, 4081),              # pieces of 4096 limbs: nearly all of a piece is overlap
    (1 << 13, 3 * 4096, 4096),
    (1 << 14, 70001, 129),
    (3 << 12, 60001, 2047),              # 3 2^k points
    (3 << 13, 50003, 6000),
])
@pytest.mark.parametrize("cfg", [dict(), dict(nprimes=4), dict(par=0)])
@pytest.mark.parametrize("top", [False, True])
def test_pieces(pieces, points, na, nb, cfg, top):
    """top: operands and x of limbs B - 1, whose carries run through every block"""
    a, s = O.gen_limbs(na, na + nb)
    b, s = O.gen_limbs(nb, s)
    x, s = O.gen_limbs(na + nb - 5, s)
    if top:
        a[:] = TOP; b[:] = TOP; x[:] = TOP
    say("pieces", points, na, nb, cfg, top)
    lib = pieces(points, **cfg)
    da, db, dx = dev(a), dev(b), dev(x)
    want, wantx = O.mul_school(a, b), O.mul_school(a, b, x)
    assert np.array_equal(host(lib.mul(da, db)), want)
    assert np.array_equal(host(lib.mul(db, da)), want)
    assert np.array_equal(host(lib.mul_add(da, db, dx)), wantx)


@pytest.mark.parametrize("na,nb", [(5000003, 300007), (1 << 21, 100), (300007, 3000017), (20000001, 70000)])
@pytest.mark.parametrize("cfg", [dict(), dict(par=0), dict(tile_log=12, pts=8)])
def test_long(pieces, na, nb, cfg):
    """the rule's own choice, and each prime by itself, against the whole transform"""
    a, s = O.gen_limbs(na, na ^ nb)
    b, _ = O.gen_limbs(nb, s)
    da, db = dev(a), dev(b)
    say("long", na, nb, cfg)
    got = host(pieces(**cfg).mul(da, db))
    assert np.array_equal(got, host(pieces(0, **cfg).mul(da, db)))
    assert O.tref_res(a, b, got)


@pytest.mark.parametrize("w", [1, 2048, 8100, 8192, 30000, 32110])
def test_cut(pieces, w):
    """only the low w limbs"""
    a, s = O.gen_limbs(30011, 5)
    b, _ = O.gen_limbs(2100, s)
    say("cut", w)
    lib = pieces(1 << 13)
    got = host(lib.mul_cut(dev(a), dev(b), 0, w))
    assert np.array_equal(got[:w], O.mul_school(a, b)[:w])
