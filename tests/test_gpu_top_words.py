"""Values within 2^52 of 2^63 in the conditional subtraction (modarith.h
csub_n), which as double-precision patterns are NaNs: forward and inverse
transforms of the largest modulus whose values get there."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logn", [5, 10, 13, 14, 16, 18])
def test_values_near_2_63(logn):
    n = 1 << logn
    q = O.primes_ntt(1 << 61, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    # 4q - 2 and 4q - 4 are in the band, and 2q - 2 as close below 2q
    assert (1 << 63) - (1 << 52) <= 4 * q - 4 < 4 * q < 1 << 63
    ctx = V.Context()
    t = V.NttTables(n, q, w)
    # Forward: the first stage's product is q - 1 in the first quarter, its sum
    # 2q - 2; the second stage's product is 0, its difference 4q - 2, which the
    # third stage subtracts 2q from.
    quarter = n // 4
    a = np.zeros(n, dtype=np.uint64)
    a[:quarter] = q - 1
    a[2 * quarter:3 * quarter] = (q - 1) * pow(w, -(n // 2), q) % q
    # Inverse: sums of words q - 1 are 2q - 2, their sums 4q - 4.
    b = np.full(n, q - 1, dtype=np.uint64)
    va, vb, f, g = ctx.from_array(a), ctx.from_array(b), ctx.vector(n), ctx.vector(n)
    va.forward_transform(f, t)
    vb.inverse_transform(g, t)
    wf, wi = O.ntt_forward(a, q, w), O.ntt_inverse(b, q, w)
    assert np.array_equal(f.read(), wf)
    assert np.array_equal(g.read(), wi)
    batch = V.Batch(ctx)
    batch.add(V.JOB_NTT_FWD, va, None, f, [t])
    batch.add(V.JOB_NTT_INV, vb, None, g, [t])
    batch.run()
    assert np.array_equal(f.read(), wf)
    assert np.array_equal(g.read(), wi)
    batch.close()
    for v in (va, vb, f, g):
        v.close()
    t.close()
    ctx.close()
