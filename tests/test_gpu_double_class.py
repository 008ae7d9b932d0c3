"""The double-precision modulus class (q < 2^50, csrc/ntt_fp.h) where its
exactness and its dispatch can go wrong: the largest modulus it takes and the
smallest one past it, inputs at the ends of their range, and forward words
that are no residues (below 2^52: reduced in doubles; above: the integer first
stage), at one-tile and two-pass sizes.  Words must equal the oracle's.
"""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context()
    yield c
    c.close()


def _moduli(n):
    below = O.primes_ntt(1 << 50, 2 * n, 1)[0]
    q = (1 << 50) + 1
    while not O.is_prime(q):
        q += 2 * n
    return below, q


def _inputs(n, q, seed):
    rng = np.random.default_rng(seed)
    top = np.full(n, q - 1, dtype=np.uint64)
    alt = np.where(np.arange(n) % 2 == 0, np.uint64(0), np.uint64(q - 1))
    wide = rng.integers(0, 1 << 52, n, dtype=np.uint64)
    edge = O.fill_uniform(n, q, seed)
    edge[rng.integers(0, n, 4)] = np.array([q, (1 << 52) - 1, 1 << 52, (1 << 64) - 1],
                                           dtype=np.uint64)
    return {"top": top, "alternating": alt, "below 2^52": wide, "edge words": edge}


@pytest.mark.parametrize("logn", [3, 8, 9, 12, 13, 14, 15, 16, 17, 18, 20])
def test_double_class_edges(ctx, logn):
    n = 1 << logn
    for q in _moduli(n):
        w = O.root_2n(q, n)
        t = V.NttTables(n, q, w)
        for name, x in _inputs(n, q, logn).items():
            a, f = ctx.from_array(x), ctx.vector(n)
            a.forward_transform(f, t)
            want = O.ntt_forward(x, q, w)
            assert np.array_equal(f.read(), want), (logn, q, name)
            if x.max() < q:
                a.inverse_transform(f, t)
                assert np.array_equal(f.read(), O.ntt_inverse(x, q, w)), (logn, q, name)
            a.close()
            f.close()
        t.close()


@pytest.mark.parametrize("logn", [3, 10, 13, 15, 19])
def test_double_class_products(ctx, logn):
    """Products mix both classes in one batch, with operands of extreme
    residues and of words past 2^52."""
    n = 1 << logn
    qs = _moduli(n)
    ws = [O.root_2n(q, n) for q in qs]
    tabs = [V.NttTables(n, q, w) for q, w in zip(qs, ws)]
    rng = np.random.default_rng(logn)
    a = np.concatenate([_inputs(n, q, 1)["top"] for q in qs])
    b = np.concatenate([_inputs(n, q, 2)["edge words"] for q in qs])
    b[:n // 2] = rng.integers(0, 1 << 63, n // 2, dtype=np.uint64)
    va, vb, r = ctx.from_array(a), ctx.from_array(b), ctx.vector(2 * n)
    batch = V.Batch(ctx)
    batch.add(V.JOB_POLYMUL, va, vb, r, tabs)
    batch.run()
    got = r.read()
    for i, (q, w) in enumerate(zip(qs, ws)):
        s = slice(i * n, (i + 1) * n)
        want = O.ntt_inverse(O.elemmul(O.ntt_forward(a[s], q, w), O.ntt_forward(b[s], q, w),
                                       q), q, w)
        assert np.array_equal(got[s], want), (logn, q)
    batch.close()
    for v in (va, vb, r):
        v.close()
    for t in tabs:
        t.close()
