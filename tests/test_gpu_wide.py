"""One-pass n = 2^14 transforms of the double-precision class with 32 words
per thread (csrc/ntt_wide.h): the largest modulus of the class and a small
one, words at the ends of their range and words that are no residues, the
RNS operations fused into the transforms.  Words must equal the oracle's.
"""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu

N = 1 << 14
# enough polynomials that an untuned batch takes these kernels on 256 CUs
COUNT = 384


@pytest.fixture(scope="module")
def ctx():
    c = V.Context()
    yield c
    c.close()


def _inputs(q):
    rng = np.random.default_rng(q)
    edge = O.fill_uniform(N, q, 1)
    edge[rng.integers(0, N, 4)] = np.array([q, (1 << 52) - 1, 1 << 52, (1 << 64) - 1],
                                           dtype=np.uint64)
    return [O.fill_uniform(N, q, 2), np.full(N, q - 1, dtype=np.uint64),
            np.where(np.arange(N) % 2 == 0, np.uint64(0), np.uint64(q - 1)),
            np.zeros(N, dtype=np.uint64), rng.integers(0, 1 << 52, N, dtype=np.uint64), edge]


@pytest.mark.parametrize("bits", [50, 30, 17])
def test_wide_batch(ctx, bits):
    q = O.primes_ntt(1 << bits, 2 * N, 1)[0]
    w = O.root_2n(q, N)
    t = V.NttTables(N, q, w)
    inputs = _inputs(q)
    words = np.concatenate([inputs[i % len(inputs)] for i in range(COUNT)])
    a, f, g = ctx.from_array(words), ctx.vector(words.size), ctx.vector(words.size)
    batch = V.Batch(ctx)
    views = [(a.view(i * N, N), f.view(i * N, N), g.view(i * N, N)) for i in range(COUNT)]
    for x, y, z in views:
        batch.add(V.JOB_NTT_FWD, x, None, y, [t])
        batch.add(V.JOB_NTT_INV, x, None, z, [t])
    batch.run()
    # in place, on both sides of the count the rule draws the line at
    for count in (256, 257):
        h = ctx.from_array(words[:N * count])
        again = V.Batch(ctx)
        again.add(V.JOB_NTT_FWD, h, None, h, [t] * count)
        again.run()
        assert np.array_equal(h.read(), f.read(0, N * count))
        again.close()
        h.close()
    got_f, got_i = f.read().reshape(COUNT, N), g.read().reshape(COUNT, N)
    for j, x in enumerate(inputs):
        want = O.ntt_forward(x, q, w)
        assert all(np.array_equal(r, want) for r in got_f[j::len(inputs)]), (bits, j)
        if x.max() < q:
            want = O.ntt_inverse(x, q, w)
            assert all(np.array_equal(r, want) for r in got_i[j::len(inputs)]), (bits, j)


@pytest.mark.parametrize("p", [2, 65537])
def test_wide_fused_operations(ctx, p):
    """INTT with the centered lift, and NTT-form rescaling (its lift and its
    scaling), against the same jobs as pointwise and transform steps."""
    qs = O.primes_ntt(1 << 50, 2 * N, 2)
    tabs = [V.NttTables(N, q, O.root_2n(q, N)) for q in qs]
    a = np.concatenate([O.fill_uniform(N, q, 5 + i) for i, q in enumerate(qs)])
    count = COUNT
    va = ctx.from_array(a)
    res, low = ctx.vector(2 * N * count), ctx.vector(N * count)
    batch = V.Batch(ctx)
    for i in range(count):
        batch.add_rns(V.JOB_INTT_CENTER, va, res.view(2 * N * i, 2 * N), tabs, [p])
        batch.add_rns(V.JOB_RESCALE_NTT, va, low.view(N * i, N), tabs)
    batch.run()
    got, gl = res.read().reshape(count, 2 * N), low.read().reshape(count, N)
    inv = [O.ntt_inverse(a[i * N:(i + 1) * N], q, O.root_2n(q, N)) for i, q in enumerate(qs)]
    want = np.concatenate([O.elemmod(x, p, q) for x, q in zip(inv, qs)])
    assert all(np.array_equal(r, want) for r in got)
    q, ql = int(qs[0]), int(qs[1])
    lift = [(int(x) - ql if int(x) > ql // 2 else int(x)) % q for x in inv[1]]
    y = O.ntt_forward(np.array(lift, dtype=np.uint64), q, O.root_2n(q, N))
    s = pow(ql, -1, q)
    want = np.array([(int(u) - int(v)) * s % q for u, v in zip(a[:N], y)], dtype=np.uint64)
    assert all(np.array_equal(r, want) for r in gl)
