"""The transform primitives convert canonical residues in their first and last pass: every pass shape on either side
(streamed rows of 1 to 9 bits, the fixed and the generic contiguous tiles, single-pass transforms, tiles of several
transforms, odd batches), residues at the ends of the range, y sharing memory with x, and a CRT whose result lies over its
planes."""
import numpy as np
import pytest

import oracle as O
from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


def residues(p, shape, seed):
    x = np.random.default_rng(seed).integers(0, p, shape, dtype=np.uint64)
    flat = x.reshape(-1)
    flat[0], flat[-1] = 0, p - 1
    return x


@pytest.mark.parametrize("logn,batch", [(1, 3), (2, 1), (3, 5), (4, 2), (7, 3), (9, 16), (10, 8), (10, 3), (11, 4), (12, 1),
                                        (12, 2), (12, 3), (13, 1), (13, 3), (14, 1), (15, 2), (16, 1), (17, 1), (18, 1),
                                        (19, 1), (20, 1), (21, 1), (22, 1)])
@pytest.mark.parametrize("r3", [False, True])
def test_transforms(nttm, logn, batch, r3):
    if r3 and logn > 20:
        pytest.skip("the radix-3 layer is the same at every length")
    prime = (logn + batch) % 4
    p, n = nttm.prime(prime), (3 if r3 else 1) << logn
    w = (nttm.root3 if r3 else nttm.root)(prime, logn)
    fwd, inv, pw = (nttm.ntt_fwd3, nttm.ntt_inv3, nttm.ntt_inv3_pw) if r3 else (nttm.ntt_fwd, nttm.ntt_inv, nttm.ntt_inv_pw)
    ofwd, oinv = (O.ntt3_fwd, O.ntt3_inv) if r3 else (O.ntt_fwd, O.ntt_inv)
    x = residues(p, (batch, n), logn)
    say("residues", logn, batch, r3)
    t = dev(x.reshape(-1))
    fwd(prime, t, logn, batch)
    X = host(t).reshape(batch, n)
    assert X.max() < p and np.array_equal(X[0], ofwd(x[0], p, w)) and np.array_equal(X[-1], ofwd(x[-1], p, w))
    inv(prime, t, logn, batch)
    assert np.array_equal(host(t).reshape(batch, n), x)

    def product(u, v):
        return oinv((u.astype(object) * v % p).astype(np.uint64), p, w)
    # y in place of its own, then y = x (a square), one of x's own transforms for all, x's first half for the pairs
    for ymode in range(3):
        rows = (batch, 1, (batch + 1) // 2)[ymode]
        pick = (lambda i: i, lambda i: 0, lambda i: i // 2)[ymode]
        y = residues(p, (rows, n), 7 + ymode)
        dy = dev(y.reshape(-1))
        t = dev(X.reshape(-1))
        pw(prime, t, dy, ymode, logn, batch)
        got = host(t).reshape(batch, n)
        for i in {0, batch - 1}:
            assert np.array_equal(got[i], product(X[i], y[pick(i)])), ymode
        assert np.array_equal(host(dy).reshape(rows, n), y)
        t = dev(X.reshape(-1))
        first = batch - rows                                          # y inside x: its last rows
        pw(prime, t, t[first * n:], ymode, logn, batch)
        got = host(t).reshape(batch, n)
        for i in {0, batch - 1}:
            assert np.array_equal(got[i], product(X[i], X[first + pick(i)])), ("shared", ymode)


@pytest.mark.parametrize("np_", [3, 4])
@pytest.mark.parametrize("n", [1, 5, 2047, 2048, 5000])
def test_crt_over_its_planes(nttm, np_, n):
    import ctypes as C
    import torch
    ps = [nttm.prime(i) for i in range(np_)]
    planes = [residues(p, (n,), i)[:n] for i, p in enumerate(ps)]
    nc = n + 4
    want = host(nttm.crt([dev(q) for q in planes], n, nc))
    M = 1
    for p in ps:
        M *= p
    v = 0
    for k in range(n - 1, -1, -1):
        v = v * O.B + sum(int(q[k]) * (M // p) * pow(M // p, -1, p) for q, p in zip(planes, ps)) % M
    assert [int(x) for x in want] == [v // O.B ** i % O.B for i in range(nc)] if n <= 5 else True
    for over in range(np_):
        buf = torch.zeros(nc, dtype=torch.int64, device="cuda")
        t = [dev(q) for q in planes]
        buf[:n] = t[over]
        t[over] = buf
        arr = (C.c_void_p * np_)(*[q.data_ptr() for q in t])
        say("crt over", np_, n, over)
        assert nttm.lib().nttm_crt(C.c_void_p(buf.data_ptr()), nc, arr, np_, n, None, 0, None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(host(buf), want)
