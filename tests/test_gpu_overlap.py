"""A result that shares memory with its own added operand x, at the same address and shifted against it: single products,
batches, plans, the one-call-each forms, the CRT primitive and empty operands, at the lengths of every kernel that reads x
(one-kernel products, the CRT with and without the last inverse pass, pieces, segments).  Against the oracle, limb for limb,
or (long products) against the same product with x elsewhere."""
import os

import numpy as np
import pytest

import oracle as O
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib(nttm):
    import torch

    def set_(points=None, **cfg):
        if points is None:
            os.environ.pop("NTTM_PIECES", None)
        else:
            os.environ["NTTM_PIECES"] = str(points)
        torch.cuda.synchronize()
        nttm.shutdown()
        nttm.init(0, **cfg)
        return nttm
    yield set_
    set_()


def shared(x, nc, shift):
    """x and a result of nc limbs in one buffer, the result `shift` limbs above x"""
    import torch
    xo, co = max(0, -shift), max(0, shift)
    buf = torch.full((max(xo + len(x), co + nc) + 8,), -1, dtype=torch.int64, device="cuda")
    buf[xo:xo + len(x)] = dev(x)
    return buf[xo:xo + len(x)], buf[co:co + nc]


# coefficients: one kernel; 2^13 points; 2^14; 2^16; more; pieces and segments (points of NTTM_PIECES)
CASES = [(40, 25, None), (2500, 1500, None), (2600, 2401, None), (3500, 3501, None), (7000, 7001, None),
         (20011, 19990, None), (100003, 99998, None), (60000, 300, None), (30011, 2100, 1 << 13), (50003, 6000, 3 << 13),
         (30011, 2100, 1 << 12), (30011, 2100, 0)]


@pytest.mark.parametrize("na,nb,points", CASES)
@pytest.mark.parametrize("cfg", [dict(), dict(nprimes=4)])
def test_result_over_x(lib, na, nb, points, cfg):
    a, s = O.gen_limbs(na, na)
    b, s = O.gen_limbs(nb, s)
    x, _ = O.gen_limbs(na + nb, s)
    say("c over x", na, nb, points, cfg)
    n = lib(points, **cfg)
    da, db = dev(a), dev(b)
    nc = na + nb + 1
    if na * nb < 500_000_000:
        want = O.mul_school(a, b, x)
    else:
        want = host(n.mul_add(da, db, dev(x)))
    ncn = int(np.nonzero(want)[0][-1]) + 1
    shifts = (0, 1, 5, -5, 64, 2048, na + nb - 3)
    for sh in shifts:
        dx, c = shared(x, nc, sh)
        n.mul_add(da, db, dx, out=c)
        assert np.array_equal(host(c), want), sh
    for call in (n.mul_batch, n.mul_each, n.mul_each_async):
        items = [(da, db) + shared(x, nc, sh) for sh in shifts] + [(db, da) + shared(x, nc, 0)]
        prods = call(n.make_prods(items))
        for it, p in zip(items, prods):
            assert np.array_equal(host(it[3]), want) and p.ncn == ncn
    items = [(da, db) + shared(x, nc, sh) for sh in shifts]
    for tune in (0, 1):
        plan = n.BatchPlan(n.make_prods(items), autotune=tune)
        for _ in range(3):
            for it in items:
                it[3].fill_(-1)
                it[2].copy_(dev(x))
            plan.run()
            assert list(plan.ncn()) == [ncn] * len(items)
            for it in items:
                assert np.array_equal(host(it[3]), want)
        plan.close()


def test_many_and_empty(lib):
    """more products than one copy launch holds, empty operands and x elsewhere among them; with the residue post-condition
    too"""
    import torch
    rng = np.random.default_rng(3)
    for check in (0, 1):
        say("many over x", check)
        n = lib(check=check)
        ops, s = [], 17
        for i in range(75):
            na, nb = int(rng.integers(1, 9000)), 0 if i % 9 == 4 else int(rng.integers(1, 4000))
            a, s = O.gen_limbs(na, s)
            b, s = O.gen_limbs(nb, s) if nb else (np.empty(0, dtype=np.uint64), s)
            x, s = O.gen_limbs(int(rng.integers(1, na + nb + 1)), s)
            ops.append((a, b, x))

        def want(a, b, x):
            if len(b):
                return O.mul_school(a, b, x)
            return np.concatenate([x, np.zeros(len(a) + 1 - len(x), dtype=np.uint64)])

        def item(i, a, b, x):
            if i % 4 == 1:
                return (dev(a), dev(b), dev(x), torch.full((len(a) + len(b) + 1,), -1, dtype=torch.int64, device="cuda"))
            return (dev(a), dev(b)) + shared(x, len(a) + len(b) + 1, (0, 3, -2)[i % 3])
        wants = [want(*o) for o in ops]
        for call in (n.mul_batch, n.mul_each, n.mul_each_async):
            items = [item(i, *o) for i, o in enumerate(ops)]
            prods = call(n.make_prods(items))
            for it, w, p in zip(items, wants, prods):
                assert np.array_equal(host(it[3]), w) and p.ncn == int(np.nonzero(w)[0][-1]) + 1
        items = [item(i, *o) for i, o in enumerate(ops)]
        plan = n.BatchPlan(n.make_prods(items), autotune=0)
        for it, o in zip(items, ops):
            it[2].copy_(dev(o[2]))
        plan.run()
        for it, w in zip(items, wants):
            assert np.array_equal(host(it[3]), w)
        plan.close()


@pytest.mark.parametrize("na,nb", [(40, 25), (3500, 3501), (30011, 2100)])
def test_chain(lib, na, nb):
    """the one-call-each forms over one accumulator: every product adds to what the one before it left"""
    import torch
    n, s = lib(), 5
    x, s = O.gen_limbs(na + nb, s)
    ops, want = [], x
    for i in range(4):
        a, s = O.gen_limbs(na, s)
        b, s = O.gen_limbs(nb, s)
        ops.append((dev(a), dev(b)))
        want = O.mul_school(a, b, want[:na + nb])
    say("chain over x", na, nb)
    for call in (n.mul_each, n.mul_each_async):
        buf = torch.zeros(na + nb + 1, dtype=torch.int64, device="cuda")
        buf[:na + nb] = dev(x)
        call(n.make_prods([(a, b, buf[:na + nb], buf) for a, b in ops]))
        assert np.array_equal(host(buf), want)


@pytest.mark.parametrize("shift", [0, 7, -7])
def test_grid_and_crt(lib, shift):
    """a grid under a workspace cap, and the CRT primitive"""
    import ctypes as C
    a, s = O.gen_limbs(9000, 5)
    b, s = O.gen_limbs(8000, s)
    x, _ = O.gen_limbs(17000, s)
    say("grid and crt over x", shift)
    n = lib(workspace_bytes=300000)
    want = O.mul_school(a, b, x)
    dx, c = shared(x, 17001, shift)
    n.mul_add(dev(a), dev(b), dx, out=c)
    assert np.array_equal(host(c), want)
    n = lib()
    N = 1 << 15
    planes = []
    for i in range(3):
        import torch
        pa, pb = torch.zeros(N, dtype=torch.int64, device="cuda"), torch.zeros(N, dtype=torch.int64, device="cuda")
        n.load(i, pa, dev(a)); n.load(i, pb, dev(b))
        n.ntt_fwd(i, pa, 15); n.ntt_fwd(i, pb, 15)
        n.ntt_inv_pw(i, pa, pb, n.Y_FULL, 15)
        planes.append(pa)
    dx, c = shared(x, 17001, shift)
    arr = (C.c_void_p * 3)(*[p.data_ptr() for p in planes])
    rc = n.lib().nttm_crt(C.c_void_p(c.data_ptr()), 17001, arr, 3, 16999, C.c_void_p(dx.data_ptr()), 17000, None)
    assert rc == 0, n.lib().nttm_last_error()
    assert np.array_equal(host(c), want)
