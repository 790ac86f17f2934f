"""The launch schedules of a product give one result: every prime and both operands in one launch per pass, or prime
after prime (NTTM_PAR_POINTS=0), and a batch group whole or in chunks through the same planes (NTTM_CHUNK_POINTS), with
shared B operands inside a chunk and across chunks, radix-3 lengths and four primes.  Products are compared with the
oracle, limb for limb."""
import os

import numpy as np
import pytest

import oracle as O
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture
def schedule(nttm):
    import torch

    def set_(par=None, chunk=None, inv_crt=None, **cfg):
        for k, v in (("NTTM_PAR_POINTS", par), ("NTTM_CHUNK_POINTS", chunk), ("NTTM_INV_CRT_POINTS", inv_crt)):
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


# a single pass, two passes at the smallest strided rows, 9-bit rows, three passes with deferred twiddles, 3 2^k
@pytest.mark.parametrize("na,nb", [(2049, 2047), (4097, 1), (5000, 3193), (700001, 300001), (1 << 21, 2097151)])
@pytest.mark.parametrize("cfg", [dict(), dict(radix3=2), dict(nprimes=4), dict(tile_log=12, pts=8)])
def test_product_schedules(schedule, na, nb, cfg):
    a, s = O.gen_limbs(na, na + nb)
    b, _ = O.gen_limbs(nb, s)
    da, db = dev(a), dev(b)
    say("schedules", na, nb, cfg)
    together = host(schedule(**cfg).mul(da, db))
    apart = host(schedule(par=0, **cfg).mul(da, db))
    assert np.array_equal(together, apart)
    if na * nb <= 20_000_000:
        assert np.array_equal(together, O.mul_school(a, b))
    else:
        assert O.tref_res(a, b, together)


@pytest.mark.parametrize("chunk", [1, 3 << 13, 1 << 15, 1 << 17])
@pytest.mark.parametrize("cfg", [dict(), dict(radix3=2)])
def test_group_chunks(schedule, chunk, cfg):
    """11 products of about 2^14 points and 7 of about 2^12, most in pairs with one B: chunks of one product, of an odd
    number of them (a pair split between two chunks) and of all"""
    import torch
    rng = np.random.default_rng(chunk)
    ops, s = [], 99
    for i in range(18):
        lo, hi = (7000, 9000) if i < 11 else (1500, 2100)
        a, s = O.gen_limbs(int(rng.integers(lo, hi)), s)
        if i % 2 == 0:
            b, s = O.gen_limbs(int(rng.integers(lo - 1000, hi - 1000)), s)
            db = dev(b)
        x = None
        if i % 3 == 0:
            x, s = O.gen_limbs(int(rng.integers(1, len(a) + len(b) + 1)), s)
        ops.append((a, b, x, db))
    say("chunks", chunk, cfg)
    n = schedule(chunk=chunk, **cfg)
    items = [(dev(a), db, None if x is None else dev(x),
              torch.full((len(a) + len(b) + (x is not None),), -1, dtype=torch.int64, device="cuda"))
             for a, b, x, db in ops]
    prods = n.make_prods(items)
    n.mul_batch(prods)
    plan = n.BatchPlan(prods, autotune=False)
    eager = [host(it[3]) for it in items]
    for _ in range(2):
        for it in items:
            it[3].fill_(-1)
        plan.run()
        lens = plan.ncn()
        for (a, b, x, _), it, c, ln, pr in zip(ops, items, eager, lens, prods):
            want = O.mul_school(a, b, x)
            assert np.array_equal(c, want) and np.array_equal(host(it[3]), want)
            assert ln == pr.ncn == int(np.nonzero(want)[0][-1]) + 1
    plan.close()


@pytest.mark.parametrize("n", [100, 5000, 300000])
@pytest.mark.parametrize("par", [None, 0])
def test_phase_times(schedule, n, par):
    """the phase times of a call are its own: none negative, together positive and within the call's wall time (plus
    the 0.01 ms tick of the device clock per phase)"""
    import time
    import torch
    lib = schedule(par=par)
    a, s = O.gen_limbs(n, 3)
    da, db = dev(a), dev(O.gen_limbs(n, s)[0])
    lib.mul(da, db)
    for _ in range(3):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        lib.mul(da, db)
        wall = 1e3 * (time.perf_counter() - t0)
        ph = lib.last_phase_ms()
        say("phases", n, par, ph, wall)
        assert all(p >= 0 for p in ph) and 0 < sum(ph) <= wall + 0.03


# pieces (NTTM_PIECES points), segments, by the rule
@pytest.mark.parametrize("points,na,nb", [(1 << 13, 1 << 18, 1), (None, 1000000, 1000), (1 << 12, 30011, 2100)])
def test_phase_times_uneven(schedule, points, na, nb):
    """an uneven product's short operand is transformed once (here for at most a 64th of the points, or in every workgroup of
    segments): its phase is above 0 and, in pieces, below a 20th of the whole; every phase has a share"""
    import time
    import torch
    if points:
        os.environ["NTTM_PIECES"] = str(points)
    try:
        lib = schedule()
    finally:
        os.environ.pop("NTTM_PIECES", None)
    a, s = O.gen_limbs(na, 3)
    da, db = dev(a), dev(O.gen_limbs(nb, s)[0])
    lib.mul(da, db)
    for _ in range(3):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        lib.mul(da, db)
        wall = 1e3 * (time.perf_counter() - t0)
        ph = lib.last_phase_ms()
        say("phases uneven", points, na, nb, ph, wall)
        assert all(p > 0 for p in ph) and sum(ph) <= wall + 0.03
        if nb == 1:
            assert ph[0] < sum(ph) / 20
        lib.mul(db, da)
        assert all(p > 0 for p in lib.last_phase_ms())


def _limbs(kind, n, s):
    if kind == "max":
        return np.full(n, O.B - 1, dtype=np.uint64), s
    if kind == "zero":
        return np.zeros(n, dtype=np.uint64), s
    return O.gen_limbs(n, s)


# around every length of the one-kernel products (2^7 .. 2^12 points) and just above the longest
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097])
@pytest.mark.parametrize("nprimes", [0, 4])
def test_one_kernel_products(schedule, n, nprimes):
    """c = a b and c = a b + x with n coefficients: random limbs, all limbs B - 1 (carry chains through every word),
    zeros, x of every length class, the low limbs alone (a cut), c over a; singly and as one batch with neighbours of
    the same kernel, an incomplete last block among them"""
    import torch
    lib = schedule(nprimes=nprimes)
    ops, s = [], n
    for kind in ("random", "max", "zero"):
        for na in sorted({1, (n + 1) // 2, n}):
            nb = n + 1 - na
            a, s = _limbs(kind, na, s)
            b, s = _limbs("random" if kind == "zero" else kind, nb, s)
            for nx in (None, 1, n, n + 1):
                x = None if nx is None else _limbs("random" if kind == "random" else "max", nx, s)[0]
                ops.append((a, b, x))
    say("one kernel", n, nprimes)
    want = [O.mul_school(a, b, x) for a, b, x in ops]
    items = [(dev(a), dev(b), None if x is None else dev(x),
              torch.full((len(w),), -1, dtype=torch.int64, device="cuda")) for (a, b, x), w in zip(ops, want)]
    prods = lib.make_prods(items)
    lib.mul_batch(prods)
    plan = lib.BatchPlan(prods, autotune=False)
    for run in (lambda: None, plan.run):
        run()
        for it, w, pr in zip(items, want, prods):
            nz = np.nonzero(w)[0]
            assert np.array_equal(host(it[3]), w) and pr.ncn == (int(nz[-1]) + 1 if len(nz) else 0)
            it[3].fill_(-1)
    assert plan.ncn() == [pr.ncn for pr in prods]
    plan.close()
    for (a, b, x), it, w in list(zip(ops, items, want))[::3]:
        got = lib.mul(it[0], it[1]) if x is None else lib.mul_add(it[0], it[1], it[2])
        assert np.array_equal(host(got), w)
    a, b, w = ops[0][0], ops[0][1], want[0]
    for cut in sorted({1, (n + 1) // 2, n}):
        assert np.array_equal(host(lib.mul_cut(items[0][0], items[0][1], w=cut)), w[:cut])
    over = torch.full((len(w),), -1, dtype=torch.int64, device="cuda")
    over[:len(a)] = items[0][0]
    lib.mul(over[:len(a)], items[0][1], out=over)
    assert np.array_equal(host(over), w)


# blocks of 2048 limbs: within one workgroup's 64, across workgroups, beyond one look of 256 words, an odd end
@pytest.mark.parametrize("blocks,extra", [(1, 0), (63, 5), (64, 0), (65, 1), (129, 2047), (320, 0), (900, 77)])
def test_carry_through_blocks(nttm, blocks, extra):
    """1 (B^n - 1) + x: with x = 1 the carry out of the first limb runs through every block to the top, with x = 0 (and
    with x = 1 placed one limb below a limb that stops it) it does not; the same by the device addition and, for the
    sign, the subtraction"""
    import torch
    n = 2048 * blocks + extra
    one = dev(np.array([1], dtype=np.uint64))
    nines = torch.full((n,), O.B - 1, dtype=torch.int64, device="cuda")
    say("carry through", blocks, extra)
    c = nttm.mul_add(one, nines, one)
    assert int(c[n]) == 1 and int(c.count_nonzero()) == 1
    c = nttm.mul_add(one, nines, torch.zeros(1, dtype=torch.int64, device="cuda"))
    assert bool((c[:n] == O.B - 1).all()) and not bool(c[n:].any())
    for stop in {0, n // 2, n - 1}:
        b = nines.clone()
        b[stop] = 5
        b[n - 1].clamp_(min=1)
        c = nttm.mul_add(one, b, one)
        want = b.clone()
        want[:stop] = 0
        want[stop] = 6
        assert torch.equal(c[:n], want) and not bool(c[n:].any())
    r, carry = nttm.debug_addsub(nines, one, n)
    assert carry and not bool(r.any())
    r, carry = nttm.debug_addsub(nines, one, n + 1)
    assert not carry and int(r[n]) == 1 and int(r.count_nonzero()) == 1
    top = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    top[n] = 1
    r, ge = nttm.debug_addsub(top, one, n + 1, sub=True)
    assert ge and bool((r[:n] == O.B - 1).all()) and int(r[n]) == 0
    r, ge = nttm.debug_addsub(one, top, n + 1, sub=True)
    assert not ge


# transforms of 2^13 .. 2^16 points: the last inverse pass runs with the CRT, in runs of 60 limbs of rows of 4096
@pytest.mark.parametrize("n", [4097, 8191, 8192, 8193, 12289, 16384, 16385, 20481, 32767, 32768, 32769, 40961, 65535, 65536])
@pytest.mark.parametrize("nprimes", [0, 4])
def test_inverse_with_crt(schedule, n, nprimes):
    """n coefficients, random and all limbs B - 1 (carries through every run and row), + x up to the transform's last limbs
    and beyond, single, batched (chunks of one product among them) and planned; against the path without it"""
    import torch
    ops, s = [], n
    for kind in ("random", "max"):
        for na in sorted({1, n // 3 + 1, (n + 1) // 2}):
            nb = n + 1 - na
            a, s = _limbs(kind, na, s)
            b, s = _limbs(kind, nb, s)
            for nx in (None, 1, n + 1):
                ops.append((a, b, None if nx is None else _limbs("max" if kind == "max" or nx == 1 else "random", nx, s)[0]))
    ops.append((np.array([1], dtype=np.uint64), np.full(n, O.B - 1, dtype=np.uint64), np.array([1], dtype=np.uint64)))
    say("inverse with crt", n, nprimes)
    lib = schedule(nprimes=nprimes, inv_crt=1)
    ps = [lib.prime(i) for i in range(4 if nprimes else 3)]
    want = [O.mul_ntt(a, b, ps, x) for a, b, x in ops]
    assert int(want[-1][n]) == 1 and not want[-1][:n].any()
    items = [(dev(a), dev(b), None if x is None else dev(x),
              torch.full((len(w),), -1, dtype=torch.int64, device="cuda")) for (a, b, x), w in zip(ops, want)]
    for chunk in (None, 1, 3 << 16):
        lib = schedule(nprimes=nprimes, chunk=chunk, inv_crt=1 if chunk else None)
        prods = lib.make_prods(items)
        lib.mul_batch(prods)
        for it, w, pr in zip(items, want, prods):
            assert np.array_equal(host(it[3]), w) and pr.ncn == int(np.nonzero(w)[0][-1]) + 1
            it[3].fill_(-1)
    plan = lib.BatchPlan(prods, autotune=False)
    plan.run()
    assert plan.ncn() == [pr.ncn for pr in prods]
    assert all(np.array_equal(host(it[3]), w) for it, w in zip(items, want))
    plan.close()
    for it, w in list(zip(items, want))[::2]:
        got = lib.mul(it[0], it[1]) if it[2] is None else lib.mul_add(it[0], it[1], it[2])
        assert np.array_equal(host(got), w)
    for cut in sorted({1, 60, 4096, 4097, n // 2, n}):
        assert np.array_equal(host(lib.mul_cut(items[3][0], items[3][1], w=cut)), want[3][:cut])


@pytest.mark.parametrize("logn", [7, 8, 9, 10, 11])
@pytest.mark.parametrize("over", [-1, 0, 1])
@pytest.mark.parametrize("np_", [3, 4])
def test_small_products_few_and_many(schedule, logn, over, np_):
    """batches of the largest count that takes a block per product (2^19 points), one less and one more, in ragged lengths"""
    import torch
    cnt = ((1 << 19) >> logn) + over
    rng = np.random.default_rng(logn * 10 + over)
    n = 1 << logn
    say("few and many", logn, cnt, np_)
    lib = schedule(nprimes=np_)
    flat, _ = O.gen_limbs(cnt * (n + 1), logn)
    df = dev(flat)
    out = torch.full((cnt * (n + 1),), -1, dtype=torch.int64, device="cuda")
    items, shape = [], []
    for i in range(cnt):
        total = int(rng.integers((n >> 1) + 2 if logn > 7 else 2, n + 2))       # na + nb - 1 coefficients of this length
        na = int(rng.integers(1, total))
        o = i * (n + 1)
        items.append((df[o:o + na], df[o + na:o + total], None, out[o:o + total]))
        shape.append((o, na, total))
    prods = lib.make_prods(items)
    lib.mul_batch(prods)
    got = host(out)
    for i in list(range(0, cnt, max(1, cnt // 300))) + [cnt - 1]:
        o, na, total = shape[i]
        want = O.mul_school(flat[o:o + na], flat[o + na:o + total])
        assert np.array_equal(got[o:o + total], want), (i, na, total)
        assert prods[i].ncn == int(np.nonzero(want)[0][-1]) + 1
    rest = np.ones(len(got), dtype=bool)
    for o, _, total in shape:
        rest[o:o + total] = False
    assert (got[rest] == np.uint64(2 ** 64 - 1)).all()
