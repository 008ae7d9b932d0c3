"""The double-precision class (q < 2^50) on every tile, pass mode, stage split
and row tile that can be chosen or tuned: each has rounds of its own, and so
bounds of its own at which values are reduced.  Words of the largest modulus of
the class at the ends of their range come closest to those bounds."""
import functools

import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    c = V.Context()
    yield c
    c.close()


@functools.lru_cache(maxsize=None)
def _oracle(logn):
    """(q, w, words of three polynomials, their transforms both ways)."""
    n = 1 << logn
    q = O.primes_ntt(1 << 50, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    polys = [np.full(n, q - 1, dtype=np.uint64),
             np.where(np.arange(n) % 2 == 0, np.uint64(0), np.uint64(q - 1)),
             O.fill_uniform(n, q, logn)]
    return (q, w, np.concatenate(polys),
            np.concatenate([O.ntt_forward(x, q, w) for x in polys]),
            np.concatenate([O.ntt_inverse(x, q, w) for x in polys]))


def _choices(logn):
    for tb in (11, 12, 13, 14):
        for mode in (1, 2, 3):
            for split in (0, 1):
                for tb2 in (0, 11, 12, 13, 14):
                    if mode == 2 or not (split or tb2):
                        yield tb, mode, split, tb2


def _choose(ctx, logn, tb, mode, split, tb2):
    ctx.set_tile_bits(logn, tb)
    ctx.set_pass_mode(logn, mode)
    ctx.set_split(logn, split)
    ctx.set_tile_bits2(logn, tb2)


@pytest.mark.parametrize("logn", range(12, 21))
def test_every_choice(ctx, logn):
    n = 1 << logn
    q, w, words, fwd, inv = _oracle(logn)
    t = V.NttTables(n, q, w)
    a, f, g, one = ctx.from_array(words), ctx.vector(3 * n), ctx.vector(3 * n), ctx.vector(n)
    batch = V.Batch(ctx)
    first = a.view(0, n)
    for choice in _choices(logn):
        _choose(ctx, logn, *choice)
        batch.clear()
        batch.add(V.JOB_NTT_FWD, a, None, f, [t] * 3)
        batch.add(V.JOB_NTT_INV, a, None, g, [t] * 3)
        batch.run()
        assert np.array_equal(f.read(), fwd), choice
        assert np.array_equal(g.read(), inv), choice
        first.forward_transform(one, t)
        assert np.array_equal(one.read(), fwd[:n]), choice
        first.inverse_transform(one, t)
        assert np.array_equal(one.read(), inv[:n]), choice
    batch.close()
    for v in (first, a, f, g, one):
        v.close()
    t.close()


@pytest.mark.parametrize("logn", range(12, 18))
def test_products_and_rescaling_of_every_choice(ctx, logn):
    """Against the built-in choice, whose words other tests compare with the
    oracle's."""
    n = 1 << logn
    q, w, words, _, _ = _oracle(logn)
    ql = O.primes_ntt(1 << 53, 2 * n, 1)[0]
    t, tl = V.NttTables(n, q, w), V.NttTables(n, ql, O.root_2n(ql, n))
    last = O.fill_uniform(n, ql, 5)
    a, b = ctx.from_array(words), ctx.from_array(words[::-1].copy())
    pairs = [ctx.from_array(np.concatenate([words[i * n:(i + 1) * n], last])) for i in range(3)]
    r, s = ctx.vector(3 * n), ctx.vector(3 * n)
    views = [s.view(i * n, n) for i in range(3)]
    batch, want = V.Batch(ctx), None
    for choice in [(0, 0, 0, 0)] + list(_choices(logn)):
        _choose(ctx, logn, *choice)
        batch.clear()
        batch.add(V.JOB_POLYMUL, a, b, r, [t] * 3)
        for p, v in zip(pairs, views):
            batch.add_rns(V.JOB_RESCALE_NTT, p, v, [t, tl])
        batch.run()
        got = (r.read(), s.read())
        want = want or got
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), choice
    batch.close()
    for v in views + pairs + [a, b, r, s]:
        v.close()
    for x in (t, tl):
        x.close()


@pytest.mark.parametrize("tile,count", [(0, 383), (0, 384), (14, 300)])
def test_one_pass_in_place(ctx, tile, count):
    """n = 2^14 in place, where 32 words per thread run (more polynomials than
    CUs in one pass) and below the rule."""
    n = 1 << 14
    q, w, words, fwd, inv = _oracle(14)
    t = V.NttTables(n, q, w)
    ctx.set_tile_bits(14, tile)
    many = np.tile(words, count // 3 + 1)[:n * count]
    for op, want in ((V.JOB_NTT_FWD, fwd), (V.JOB_NTT_INV, inv)):
        v = ctx.from_array(many)
        batch = V.Batch(ctx)
        batch.add(op, v, None, v, [t] * count)
        batch.run()
        assert batch.shape()[0] == (2 if (tile, count) == (0, 383) else 1)
        assert np.array_equal(v.read(), np.tile(want, count // 3 + 1)[:n * count]), (op, count)
        batch.close()
        v.close()
    t.close()
