"""Which route a batch takes, seen by its launches and branches
(vkhel_batch_shape): parallel branches only for independent steps, forward and
inverse transforms together only where they fit on the device at once, n = 2^14
in one pass by its number and class.  Counts are those of 256 CUs."""
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


def _table(ctx, logn, bits):
    n = 1 << logn
    q = O.primes_ntt(1 << bits, 2 * n, 1)[0]
    return n, q, V.NttTables.on_device(ctx, n, q, O.root_2n(q, n))


def _shape(ctx, jobs):
    """Shape of a batch of (op, a, result, tables), run once."""
    batch = V.Batch(ctx)
    for op, a, r, tabs in jobs:
        batch.add(op, a, a if op >= V.JOB_POLYMUL else None, r, tabs)
    assert batch.shape() == (0, 0)
    batch.run()
    shape = batch.shape()
    batch.close()
    return shape


def _transforms(ctx, logn, bits, nfwd, ninv):
    n, _, t = _table(ctx, logn, bits)
    a, f, g = (ctx.vector(n * max(k, 1)) for k in (max(nfwd, ninv), nfwd, ninv))
    jobs = [(V.JOB_NTT_FWD, a, f, [t] * nfwd)] if nfwd else []
    jobs += [(V.JOB_NTT_INV, a, g, [t] * ninv)] if ninv else []
    shape = _shape(ctx, jobs)
    for v in (a, f, g):
        v.close()
    t.close()
    return shape


def test_independent_steps_branch_and_dependent_ones_do_not(ctx):
    for dependent in (False, True):
        jobs, kept = [], []
        for logn in (10, 11, 12, 13, 14, 15):
            n, q, t = _table(ctx, logn, 60)
            a, f, g, m = (ctx.vector(n) for _ in range(4))
            jobs += [(V.JOB_NTT_FWD, a, f, [t]), (V.JOB_POLYMUL, a, m, [t]),
                     (V.JOB_NTT_INV, f if dependent else a, g, [t])]
            kept += [a, f, g, m, t]
        launches, branches = _shape(ctx, jobs)
        assert launches > 8 and branches == (1 if dependent else 4), (launches, branches)
        for k in kept:
            k.close()


# one launch for whole transforms, two for two passes; apart, twice as many
@pytest.mark.parametrize("logn,nfwd,ninv,launches", [
    (10, 8, 8, 1), (12, 300, 212, 1), (12, 300, 213, 2), (13, 5, 251, 1), (13, 5, 252, 2),
    (14, 100, 156, 2), (14, 100, 157, 4), (16, 33, 31, 2), (16, 33, 32, 4)])
@pytest.mark.parametrize("bits", [50, 60])
def test_both_directions_together(ctx, bits, logn, nfwd, ninv, launches):
    assert _transforms(ctx, logn, bits, nfwd, ninv) == (launches, 1)


@pytest.mark.parametrize("bits,polys,launches", [
    (50, 191, 2), (50, 192, 1), (50, 256, 1), (50, 257, 2), (50, 383, 2), (50, 384, 1),
    (50, 1025, 1), (60, 223, 2), (60, 224, 1), (60, 256, 1), (60, 257, 2), (60, 447, 2),
    (60, 448, 1), (60, 512, 1), (60, 513, 2), (60, 1024, 1), (60, 1025, 2)])
def test_one_pass_rule(ctx, bits, polys, launches):
    assert _transforms(ctx, 14, bits, polys, 0) == (launches, 1)
    assert _transforms(ctx, 14, bits, 0, polys) == (launches, 1)


def test_pass_mode_2_is_the_default(ctx):
    """Mode 2 (what the tuner names) launches what mode 0 does; mode 1 runs
    whole polynomials, both directions apart."""
    for mode, want in ((0, [1, 1, 2, 1]), (2, [1, 1, 2, 1]), (1, [2, 2, 2, 1])):
        got = []
        for logn, nfwd, ninv in ((10, 8, 8), (13, 16, 16), (16, 8, 8), (14, 256, 0)):
            ctx.set_pass_mode(logn, mode)
            got.append(_transforms(ctx, logn, 50, nfwd, ninv)[0])
        assert got == want, (mode, got)


def test_tuned_contexts_go_by_number_and_class(ctx, tmp_path):
    """One pass of n = 2^14 wins the tuner's batch; few polynomials still run
    in two passes on a tuned context, and on one that loads its choices."""
    ctx.autotune(14, 14)
    ctx.autotune_save(tmp_path / "tuned")
    loaded = V.Context()
    loaded.autotune_load(tmp_path / "tuned")
    for c in (ctx, loaded):
        assert c.tile_bits(14) != 14
        for bits in (50, 60):
            assert _transforms(c, 14, bits, 16, 0) == (2, 1)
    loaded.close()
