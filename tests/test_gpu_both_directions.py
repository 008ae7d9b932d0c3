"""Forward and inverse transforms of one size in one launch (ntt.hip
launch_both_ok): unequal numbers of both, on both sides of the rule's bound,
every size and modulus class, plain and with the centered lift; jobs that
share words keep their order."""
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


def _run(ctx, logn, bits, nfwd, ninv):
    n = 1 << logn
    q = O.primes_ntt(1 << bits, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    t = V.NttTables(n, q, w)
    a = O.fill_uniform(n, q, logn)
    b = np.where(np.arange(n) % 2 == 0, np.uint64(0), np.uint64(q - 1))
    words = np.concatenate([a, b])
    va = ctx.from_array(words)
    views = [va.view(0, n), va.view(n, n)]
    f, g, c = ctx.vector(n * nfwd), ctx.vector(n * ninv), ctx.vector(n)
    batch = V.Batch(ctx)
    for i in range(nfwd):
        batch.add(V.JOB_NTT_FWD, views[i % 2], None, f.view(i * n, n), [t])
    for i in range(ninv):
        batch.add(V.JOB_NTT_INV, views[i % 2], None, g.view(i * n, n), [t])
    batch.add_rns(V.JOB_INTT_CENTER, views[0], c, [t], [65537])
    batch.run()
    wf = [O.ntt_forward(x, q, w) for x in (a, b)]
    wi = [O.ntt_inverse(x, q, w) for x in (a, b)]
    gf, gi = f.read().reshape(nfwd, n), g.read().reshape(ninv, n)
    for i in range(nfwd):
        assert np.array_equal(gf[i], wf[i % 2]), (logn, bits, i)
    for i in range(ninv):
        assert np.array_equal(gi[i], wi[i % 2]), (logn, bits, i)
    assert np.array_equal(c.read(), O.elemmod(wi[0], 65537, q))
    batch.close()


@pytest.mark.parametrize("bits", [50, 54, 60, 61])
@pytest.mark.parametrize("logn", range(3, 21))
def test_sizes(ctx, logn, bits):
    _run(ctx, logn, bits, 3 if logn < 18 else 2, 1)


@pytest.mark.parametrize("logn,nfwd,ninv", [(12, 300, 211), (12, 300, 212), (13, 5, 250),
                                            (14, 100, 155), (14, 100, 156), (16, 33, 30),
                                            (16, 33, 31)])
def test_bound(ctx, logn, nfwd, ninv):
    _run(ctx, logn, 60, nfwd, ninv)


def test_shared_words_keep_their_order(ctx):
    for logn in (11, 14):
        n = 1 << logn
        q = O.primes_ntt(1 << 60, 2 * n, 1)[0]
        w = O.root_2n(q, n)
        t = V.NttTables(n, q, w)
        a = O.fill_uniform(n, q, 3)
        va, mid, out = ctx.from_array(a), ctx.vector(n), ctx.vector(n)
        batch = V.Batch(ctx)
        batch.add(V.JOB_NTT_INV, mid, None, out, [t])
        batch.add(V.JOB_NTT_FWD, va, None, mid, [t])
        batch.run()
        assert np.array_equal(out.read(), a)
        batch.close()
