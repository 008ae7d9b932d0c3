"""Batches of many unlike jobs run their steps as parallel branches of a graph
where no job needs another's words (csrc/batch.hip capture_branches): replayed
among other work, such a batch computes the same words every time, and a batch
whose jobs do depend on each other keeps its order."""
import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V

pytestmark = pytest.mark.gpu

SIZES = [4, 10, 11, 12, 13, 14, 15]


@pytest.fixture(scope="module")
def ctx():
    c = V.Context()
    yield c
    c.close()


def _table(logn, bits=60):
    n = 1 << logn
    q = O.primes_ntt(1 << bits, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    return n, q, w, V.NttTables(n, q, w)


def test_branches_replayed(ctx):
    batch, checks, kept = V.Batch(ctx), [], []
    for i, logn in enumerate(SIZES):
        n, q, w, t = _table(logn, 50 if i % 2 else 60)
        a, b = O.fill_uniform(n, q, 2 * i), O.fill_uniform(n, q, 2 * i + 1)
        va, vb = ctx.from_array(a), ctx.from_array(b)
        for op, want in ((V.JOB_NTT_FWD, O.ntt_forward(a, q, w)),
                         (V.JOB_NTT_INV, O.ntt_inverse(a, q, w)),
                         (V.JOB_POLYMUL, O.polymul_ntt(a, b, q, w)),
                         (V.JOB_MUL, O.elemmul(a, b, q))):
            r = ctx.vector(n)
            batch.add(op, va, vb if op >= V.JOB_POLYMUL else None, r, [t])
            checks.append((r, want))
        # in place
        v = ctx.from_array(a)
        batch.add(V.JOB_NTT_FWD, v, None, v, [t])
        kept += [va, vb, t, (v, a, q, w)]
    for _ in range(5):
        batch.run()
        for r, want in checks:
            assert np.array_equal(r.read(), want)
            r.copy_from_host(np.zeros(want.size, dtype=np.uint64))
        for k in kept:
            if isinstance(k, tuple):
                v, a, q, w = k
                assert np.array_equal(v.read(), O.ntt_forward(a, q, w))
                v.copy_from_host(a)
    batch.close()


def test_dependent_jobs_keep_their_order(ctx):
    """Forward results of every size that the same batch inverts, through
    views that share only part of a vector."""
    batch, checks = V.Batch(ctx), []
    for i, logn in enumerate(SIZES[1:]):
        n, q, w, t = _table(logn)
        a = O.fill_uniform(2 * n, q, i)
        va, mid, out = ctx.from_array(a), ctx.vector(2 * n), ctx.vector(n)
        batch.add(V.JOB_NTT_FWD, va, None, mid, [t, t])
        batch.add(V.JOB_NTT_INV, mid.view(n, n), None, out, [t])
        checks.append((out, a[n:], va, mid, t))
    for _ in range(3):
        batch.run()
        for out, want, *_ in checks:
            assert np.array_equal(out.read(), want)
            out.copy_from_host(np.zeros(want.size, dtype=np.uint64))
    batch.close()
