"""Synchronous calls (csrc/call_wait.h): calls of several threads on one context
each return with their results there, and a few calls alone leave the runtime
nothing to make up for when the program synchronises."""
import threading
import time

import numpy as np
import pytest

from oracle import oracle as O
import vkhel_amd as V
from vkhel_amd import hipstream

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context()
    yield c
    c.close()


def test_threads_on_one_context(ctx):
    """Lengths from a word to past 2^22, pointwise and transforms, every
    result copied on a stream that only the call's return orders, after runs
    of calls of which some watch and some block."""
    n = 1 << 16
    q = O.primes_ntt(1 << 50, 2 * n, 1)[0]
    w = O.root_2n(q, n)
    t = V.NttTables(n, q, w)
    failed = []

    def work(words, seed):
        x = O.fill_uniform(words, q, seed)
        a, r = ctx.from_array(x), ctx.vector(words)
        out, copies = V.HostBuffer(words), hipstream.Stream()
        want = O.ntt_forward(x, q, w) if words == n else None
        for k in range(6):
            for _ in range(24):
                if want is not None:
                    a.forward_transform(r, t)
                else:
                    a.elemgtadd(r, q // 2, k)
            r.read_async(out.array, 0, copies)
            copies.synchronize()
            if not np.array_equal(out.array, O.elemgtadd(x, q // 2, k)
                                  if want is None else want):
                failed.append((words, k))
        copies.close()
        out.close()
        for v in (a, r):
            v.close()

    threads = [threading.Thread(target=work, args=(words, i)) for i, words in enumerate(
        (1, 1000, n, n, (1 << 22) - 1, 1 << 22, (1 << 22) + 1, 3))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failed, failed
    t.close()


def test_few_calls_leave_an_idle_stream(ctx):
    """The stream is idle after four calls that were waited for: waiting for
    it costs less than one of them (it costs two where the runtime has not seen
    their kernels finish)."""
    a, r = ctx.vector(4096), ctx.vector(4096)
    calls, after = [], []
    for _ in range(60):
        time.sleep(0.001)
        t0 = time.perf_counter()
        for k in range(4):
            a.elemgtadd(r, 5, k)
        t1 = time.perf_counter()
        ctx.synchronize()
        calls.append((t1 - t0) / 4)
        after.append(time.perf_counter() - t1)
    print("call %.1f us, wait after 4: %.1f us" % (np.median(calls) * 1e6,
                                                   np.median(after) * 1e6))
    assert np.median(after) < np.median(calls)
    for v in (a, r):
        v.close()
