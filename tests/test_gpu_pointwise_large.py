"""Pointwise calls on vectors past the last-level cache (elementwise.hip
streams_past_cache), aligned and as views at an odd word, in place too,
against the oracle; lengths on both sides of the rule for two and three
vectors."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("length", [(1 << 25) // 3, (1 << 25) // 3 + 1, 1 << 24,
                                    (1 << 24) + 1])
def test_pointwise_past_the_cache(length, offset):
    ctx = V.Context()
    q = 1152921504606830593
    x, y = O.fill_uniform(length, q, 1), O.fill_uniform(length, q, 2)
    base = [ctx.vector(length + offset, False) for _ in range(3)]
    a, b, r = (v.view(offset, length) for v in base)
    a.write(x)
    b.write(y)
    a.elemmul(b, r, q)
    assert np.array_equal(r.read(), O.elemmul(x, y, q))
    a.elemfma(b, r, 3, q)
    assert np.array_equal(r.read(), O.elemfma(x, y, 3, q))
    a.elemgtsub(r, q // 2, 12345, 65537)
    assert np.array_equal(r.read(), O.elemgtsub(x, q // 2, 12345, 65537))
    a.elemgtadd(a, q // 2, 12345)  # in place
    assert np.array_equal(a.read(), O.elemgtadd(x, q // 2, 12345))
    b.elemmod(b, 65537, q)
    assert np.array_equal(b.read(), O.elemmod(y, 65537, q))
    for v in (a, b, r, *base):
        v.close()
    ctx.close()
