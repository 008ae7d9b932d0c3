"""Untuned n = 2^14 batches run in two passes or in one by their number
(ntt.hip tile_bits_for_tasks): on both sides of the rule's edges, for every
modulus class, a batch computes what the same batch with its tile set does."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [50, 54, 60, 61])
@pytest.mark.parametrize("polys", [1, 191, 192, 223, 224, 256, 257, 512])
def test_2_14_batches_either_way(polys, bits):
    ctx = V.Context()
    n = 1 << 14
    q = O.primes_ntt(1 << bits, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    t = V.NttTables(n, q, w)
    a, f, g = (ctx.vector(n * polys, False) for _ in range(3))
    a.fill_uniform(q, polys)
    x = a.read(n * (polys - 1), n)
    batch = V.Batch(ctx)
    batch.add(V.JOB_NTT_FWD, a, None, f, [t] * polys)
    batch.add(V.JOB_NTT_INV, a, None, g, [t] * polys)
    got = []
    for tile in (0, 12, 14):
        ctx.set_tile_bits(14, tile)
        batch.run()
        got.append((f.read(), g.read()))
    assert np.array_equal(got[0][0][-n:], O.ntt_forward(x, q, w))
    assert np.array_equal(got[0][1][-n:], O.ntt_inverse(x, q, w))
    for other in got[1:]:
        assert np.array_equal(got[0][0], other[0])
        assert np.array_equal(got[0][1], other[1])
    batch.close()
    for v in (a, f, g):
        v.close()
    t.close()
    ctx.close()
