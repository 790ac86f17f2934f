"""Batches and trees under a cap on the workspace (nttm_config.workspace_bytes): planes for every prime of both operands, for
fewer products at a time, and prime after prime through np + 1 planes, down to one product's, which is refused below
that.  Products against the oracle, limb for limb; a tree against the uncapped one."""
import numpy as np
import pytest

import oracle as O
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu
PLANE = 8 << 14                         # bytes of one prime's plane of a product of 2^14 points
SLACK = 16 << 10                        # beside the planes


@pytest.fixture
def capped(nttm):
    import torch

    def set_(cap=0, **cfg):
        torch.cuda.synchronize()
        nttm.shutdown()
        nttm.init(0, workspace_bytes=cap, **cfg)
        return nttm
    yield set_
    set_()


def batch_ops(n, share):
    """n products of 16384 coefficients, in pairs with one B (share)"""
    ops, s = [], n
    for i in range(n):
        a, s = O.gen_limbs(8192 + i % 3, s)
        if not share or i % 2 == 0:
            b, s = O.gen_limbs(8190, s)
            db = dev(b)
        x = O.gen_limbs(9000, s)[0] if i % 2 else None
        ops.append((a, b, x, db))
    return ops


# planes the cap has room for (3 primes): one product prime after prime (4), the two of a shared pair as they once were (7),
# one product with all planes (6), several
@pytest.mark.parametrize("planes", [4, 6, 7, 8, 13, 29])
@pytest.mark.parametrize("n,share", [(1, False), (2, True), (9, True), (5, False)])
def test_batch(capped, planes, n, share):
    import torch
    say("capped batch", planes, n, share)
    lib = capped(planes * PLANE + SLACK)
    ops = batch_ops(n, share)
    items = [(dev(a), db, None if x is None else dev(x),
              torch.full((len(a) + len(b) + (x is not None),), -1, dtype=torch.int64, device="cuda")) for a, b, x, db in ops]
    prods = lib.mul_batch(lib.make_prods(items))
    for (a, b, x, _), it, p in zip(ops, items, prods):
        want = O.mul_school(a, b, x)
        assert np.array_equal(host(it[3]), want) and p.ncn == int(np.nonzero(want)[0][-1]) + 1


def test_batch_refused(capped):
    """below one product's np + 1 planes"""
    import torch
    lib = capped(4 * PLANE - 1)
    say("refused batch")
    a, b, _, db = batch_ops(1, False)[0]
    c = torch.empty(len(a) + len(b), dtype=torch.int64, device="cuda")
    with pytest.raises(lib.NttmError) as e:
        lib.mul_batch(lib.make_prods([(dev(a), db, None, c)]))
    assert e.value.code == -2


@pytest.mark.parametrize("planes", [4, 6, 8, 13])
def test_tree(capped, planes):
    """8 leaves of 2048 limbs: the last level's two products of 16384 coefficients share their B"""
    leaves, s = [], 7
    for i in range(8):
        q, s = O.gen_limbs(2048, s)
        p, s = O.gen_limbs(2047, s)
        leaves.append((dev(p), dev(q)))
    say("capped tree", planes)
    want = [host(t) for t in capped().bs_tree(leaves)]
    got = [host(t) for t in capped(planes * PLANE + SLACK).bs_tree(leaves)]
    assert all(np.array_equal(g, w) for g, w in zip(got, want))


@pytest.mark.parametrize("cap", [40 << 20, 80 << 20])
def test_large(capped, cap):
    """2^20 points under 40 MiB (np + 1 planes take 32, all planes 48); 2^21 under 80 (64 and 96)"""
    import torch
    n = (1 << 19) if cap == 40 << 20 else 1 << 20
    a, s = O.gen_limbs(n, 3)
    b, _ = O.gen_limbs(n, s)
    say("capped large", cap)
    lib = capped(cap)
    da, db = dev(a), dev(b)
    c = torch.empty(2 * n, dtype=torch.int64, device="cuda")
    lib.mul_batch(lib.make_prods([(da, db, None, c)]))
    assert O.tref_res(a, b, host(c))
    assert np.array_equal(host(c), host(lib.mul(da, db)))


def test_device_nearly_full(capped):
    """no cap, but room on the device for np + 1 planes of 2^24 points (512 MiB) and not for 2 np (768): single, each, batch,
    plan, cyclic and tree"""
    import torch
    n = 1 << 23
    a, s = O.gen_limbs(n, 3)
    b, _ = O.gen_limbs(n, s)
    da, db, c = dev(a), dev(b), torch.empty(2 * n, dtype=torch.int64, device="cuda")
    lib = capped()
    want = lib.mul(da, db).clone()
    lib.mul_batch(lib.make_prods([(da, db, None, c)]))
    leaves = [(da[:n - 1], db), (db[:n - 1], da)]
    tree = [t.clone() for t in lib.bs_tree(leaves)]
    cyc = lib.mul_cyclic(da, db, 2 * n)
    assert torch.equal(c, want) and O.tref_res(a, b, host(want))

    def calls():
        prods = lib.make_prods([(da, db, None, c)])
        yield "mul", lambda: lib.mul(da, db, out=c), lambda: torch.equal(c, want)
        yield "each", lambda: lib.mul_each_async(prods), lambda: torch.equal(c, want)
        yield "batch", lambda: lib.mul_batch(prods), lambda: torch.equal(c, want)
        for tune in (0, 1):
            yield "plan", lambda: planned(prods, tune), lambda: torch.equal(c, want)

    def planned(prods, tune):
        plan = lib.BatchPlan(prods, autotune=tune)
        plan.run()
        plan.ncn()
        plan.close()
    most = fill(3 << 30)                                          # (once: it takes seconds)
    for name, call, ok in calls():
        lib = capped()
        c.fill_(-1)
        held = fill(640 << 20)
        say("nearly full", name, torch.cuda.mem_get_info()[0] >> 20)
        call()
        assert ok(), name
        del held
    lib = capped()
    held = fill((640 + 4 * 128 + 80) << 20)                       # (and the root's and the level's two numbers, the descriptors)
    say("nearly full tree", torch.cuda.mem_get_info()[0] >> 20)
    got = lib.bs_tree(leaves)
    assert all(torch.equal(g, w) for g, w in zip(got, tree))
    del held, got
    lib = capped()
    held = fill((640 + 130) << 20)
    say("nearly full cyclic", torch.cuda.mem_get_info()[0] >> 20)
    got = lib.mul_cyclic(da, db, 2 * n)
    assert torch.equal(got, cyc)
    del held, most
    torch.cuda.empty_cache()


def fill(leave):
    """device memory held so that about `leave` bytes are free"""
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = []
    while True:
        left = torch.cuda.mem_get_info()[0] - leave
        if left < 8 << 20:
            return held
        held.append(torch.empty(min(left, 32 << 30), dtype=torch.uint8, device="cuda"))
