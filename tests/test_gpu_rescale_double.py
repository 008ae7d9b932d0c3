"""NTT-form rescaling in the double-precision class (its epilogue runs on
doubles, csrc/ntt_fused.h fp_scale_word): every round shape's bound, extreme
words, dropped moduli below and above 2^52, against INTT of the dropped limb,
its centered lift, NTT and the scaling in exact integers."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("last_bits", [40, 50, 53, 61])
@pytest.mark.parametrize("logn", [3, 4, 5, 6, 7, 9, 12, 13, 14, 16, 18])
def test_rescale_words(logn, last_bits):
    ctx = V.Context()
    n = 1 << logn
    q = O.primes_ntt(1 << 50, 2 * n, 2)[1]
    ql = O.primes_ntt(1 << last_bits, 2 * n, 1)[0]
    w, wl = O.root_2n(q, n), O.root_2n(ql, n)
    tabs = [V.NttTables(n, q, w), V.NttTables(n, ql, wl)]
    a = O.fill_uniform(n, q, 1)
    a[:n // 4] = q - 1
    a[n // 4:n // 2] = 0
    coeff = O.fill_uniform(n, ql, 2)
    coeff[:4] = [0, ql // 2, ql // 2 + 1, ql - 1]
    last = O.ntt_forward(coeff, ql, wl)
    va, r = ctx.from_array(np.concatenate([a, last])), ctx.vector(n)
    batch = V.Batch(ctx)
    batch.add_rns(V.JOB_RESCALE_NTT, va, r, tabs)
    batch.run()
    lift = np.array([(int(c) - ql if int(c) > ql // 2 else int(c)) % q for c in coeff],
                    dtype=np.uint64)
    y = O.ntt_forward(lift, q, w)
    inv = pow(ql, -1, q)
    want = [(int(x) - int(z)) * inv % q for x, z in zip(a, y)]
    assert r.read().tolist() == want
    batch.close()
    for v in (va, r):
        v.close()
    for t in tabs:
        t.close()
    ctx.close()
