"""Batches whose first passes load their input with the nontemporal hint
(batch.hip stream_input: 2^24 words or more, none in place) give the words of
the same transforms in place, in every direction, class and split."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logn,bits", [(15, 60), (16, 50), (16, 55), (17, 61), (20, 50)])
def test_streamed_input_matches_in_place(logn, bits):
    ctx = V.Context()
    n = 1 << logn
    polys = (1 << 24 >> logn) + 1
    q = O.primes_ntt(1 << bits, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    t = V.NttTables(n, q, w)
    a, f, g = (ctx.vector(n * polys, False) for _ in range(3))
    a.fill_uniform(q, logn)
    x = a.read()
    out, place = V.Batch(ctx), V.Batch(ctx)
    out.add(V.JOB_NTT_FWD, a, None, f, [t] * polys)
    out.add(V.JOB_NTT_INV, a, None, g, [t] * polys)
    out.run()
    got_f, got_g = f.read(), g.read()
    for op, got in ((V.JOB_NTT_FWD, got_f), (V.JOB_NTT_INV, got_g)):
        a.write(x)
        place.clear()
        place.add(op, a, None, a, [t] * polys)
        place.run()
        assert np.array_equal(a.read(), got)
    assert np.array_equal(got_f[-n:], O.ntt_forward(x[-n:], q, w))
    # products: both column passes stream
    a.write(x)
    r = ctx.vector(n * polys, False)
    out.clear()
    out.add(V.JOB_POLYMUL, a, f, r, [t] * polys)
    out.run()
    want = O.polymul_ntt(x[:n], got_f[:n], q, w)
    assert np.array_equal(r.read(0, n), want)
    out.close()
    place.close()
    for v in (a, f, g, r):
        v.close()
    t.close()
    ctx.close()
