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
    (1 << 12, 32768, 1),                 # segments of the result, one launch: 4032 limbs each
    (1 << 12, 4032 * 3 - 61, 61),        # the result ends with a segment (4032 limbs) ...
    (1 << 12, 4032 * 3 - 60, 61),        # ... and a limb after it
    (1 << 12, 30011, 2100),
    (1 << 12, 9001, 3581),               # the longest short operand: 512 limbs of 4096 points
    (1 << 12, 70003, 700),
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


@pytest.mark.parametrize("points", [None, 1 << 12])
@pytest.mark.parametrize("cfg", [dict(), dict(nprimes=4)])
@pytest.mark.parametrize("top", [False, True])
def test_batch(pieces, points, cfg, top):
    """a batch, by call and as a plan, whose uneven products go through segments (by the rule, or all that can): lengths, added
    operands, several segments and products per workgroup, among products of other classes"""
    import torch
    rng = np.random.default_rng(11)
    ops, s = [], 5
    for i in range(70):
        lo, hi = ((1, 300), (9000, 40000)) if i % 3 else ((1, 3500), (1, 5000))
        na, nb = int(rng.integers(*hi)), int(rng.integers(*lo))
        a, s = O.gen_limbs(na, s)
        b, s = O.gen_limbs(nb, s)
        x = O.gen_limbs(int(rng.integers(1, na + nb + 1)), s)[0] if i % 4 == 0 else None
        if top:
            a[:] = TOP; b[:] = TOP
            if x is not None:
                x[:] = TOP
        ops.append((a, b, x) if i % 2 else (b, a, x))
    say("batch", points, cfg, top)
    lib = pieces(points, **cfg)
    want = [O.mul_school(*o) for o in ops]
    items = [(dev(a), dev(b), None if x is None else dev(x),
              torch.full((len(w),), -1, dtype=torch.int64, device="cuda")) for (a, b, x), w in zip(ops, want)]
    prods = lib.make_prods(items)
    lib.mul_batch(prods)
    lens = [int(np.nonzero(w)[0][-1]) + 1 for w in want]
    assert [p.ncn for p in prods] == lens
    for it, w in zip(items, want):
        assert np.array_equal(host(it[3]), w)
    for tune in (0, 1):
        plan = lib.BatchPlan(prods, autotune=tune)
        for _ in range(2):
            for it in items:
                it[3].fill_(-1)
            plan.run()
            assert list(plan.ncn()) == lens
            for it, w in zip(items, want):
                assert np.array_equal(host(it[3]), w)
        plan.close()


def test_result_over_operand(pieces):
    """a result that overwrites its own operand is formed by the passes, which read every limb first"""
    import torch
    a, s = O.gen_limbs(60000, 3)
    b, _ = O.gen_limbs(300, s)
    say("result over operand")
    lib = pieces()
    want = O.mul_school(a, b)
    for off in (0, 17, 4000):
        buf = torch.zeros(70000, dtype=torch.int64, device="cuda")
        buf[off:off + 60000] = dev(a)
        lib.mul(buf[off:off + 60000], dev(b), out=buf[:60300])
        assert np.array_equal(host(buf)[:60300], want)
        buf[off:off + 60000] = dev(a)
        lib.mul_batch(lib.make_prods([(buf[off:off + 60000], dev(b), None, buf[:60300])]))
        assert np.array_equal(host(buf)[:60300], want)
