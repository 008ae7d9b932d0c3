"""The end of a synchronous call: results are there when it returns, whether
the wait watches the completion word or blocks (a call behind work that takes
longer than the watch, a call of more words than it covers)."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V
from vkhel_amd import hipstream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words", [1, 1000, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("behind", [False, True])
def test_call_returns_complete(words, behind):
    ctx = V.Context()
    n, polys = 1 << 16, 256
    q = O.primes_ntt(1 << 50, 2 * n, 1)[0]
    t = V.NttTables(n, q, O.root_2n(q, n))
    slab = ctx.vector(n * polys, False)
    slab.fill_uniform(q, 3)
    batch = V.Batch(ctx)
    batch.add(V.JOB_NTT_FWD, slab, None, slab, [t] * polys)
    batch.run()
    x = O.fill_uniform(words, q, words)
    a, r = ctx.from_array(x), ctx.vector(words)
    out, copies = V.HostBuffer(words), hipstream.Stream()
    for k in range(3):
        if behind:
            for _ in range(8):  # about a millisecond ahead on the stream
                batch.launch()
        a.elemgtadd(r, q // 2, k)
        # (copied on a stream of its own: only the call's wait orders it)
        r.read_async(out.array, 0, copies)
        copies.synchronize()
        assert np.array_equal(out.array, O.elemgtadd(x, q // 2, k)), k
    copies.close()
    out.close()
    batch.close()
    for v in (slab, a, r):
        v.close()
    t.close()
    ctx.close()
