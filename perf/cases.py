"""Performance cases: what programs on this library spend their time in.

Every case goes through the public Python mirror of the C API (vkhel_amd):
the reference's synchronous per-vector calls (kinds call_*), the batch API
(kinds batch_* and mix) and the serving engine (kind serve).  Sizes are
those of the tests and of bench.py, or lie between them: n from 2^10 to
2^20, 1 to 24 limbs, moduli of 30 to 61 bits, vectors of any length.

Inputs are residues uniform in [0, q), as RNS limbs of ciphertexts are.
Outputs are the result vectors themselves, whole 64-bit words (seen as
int64 tensors); they have to be equal word for word, so there is no
rounding for exact() to measure.

Batches are enqueued (Batch.launch) the way a program that streams work
through the device does; the single calls wait, as the reference's do.
Contexts run with the built-in kernel choices, not tuned ones.
"""
import functools
import random

import torch

import vkhel_amd as V


# ------------------------------------------------------------------ cases

def listed():
    return [
        # One ciphertext-sized product through the reference's own API, one
        # synchronous call per step (forward, forward, elemmul, inverse):
        # a program written for the reference, relinked.  Call latency.
        {"name": "call_polymul_4096", "kind": "call_polymul", "logn": 12, "bits": 60},
        # A single two-pass transform each way: the per-call path at the
        # largest ring degree in common use.
        {"name": "call_ntt_65536", "kind": "call_ntt", "logn": 16, "bits": 50},
        # The five pointwise calls on one 24-limb RNS polynomial of odd
        # total length (a view that is not a multiple of anything).
        {"name": "call_pointwise_rns", "kind": "call_pointwise", "words": 24 * 32768 + 1,
         "bits": 60},
        # The same on vectors far larger than the caches: streaming rate.
        {"name": "call_pointwise_large", "kind": "call_pointwise", "words": 100000007,
         "bits": 55},
        # One ciphertext (two polynomials of 8 limbs) there and back: the
        # ordinary size of an evaluator that does one operation at a time,
        # too small to fill the device.
        {"name": "batch_ntt_ciphertext", "kind": "batch_ntt", "logn": 13, "limbs": 8,
         "polys": 2, "bits": 60},
        # Many small rings in one batch (one pass over memory per
        # transform, bound by the arithmetic).
        {"name": "batch_ntt_4096", "kind": "batch_ntt", "logn": 12, "limbs": 4, "polys": 2048,
         "bits": 60},
        # 64 polynomials per modulus, 8 moduli below 2^50, forward and
        # inverse, at the two ring degrees of the batched benchmark.
        {"name": "batch_ntt_16384", "kind": "batch_ntt", "logn": 14, "limbs": 8, "polys": 64,
         "bits": 50},
        {"name": "batch_ntt_65536", "kind": "batch_ntt", "logn": 16, "limbs": 8, "polys": 64,
         "bits": 50},
        # Products of polynomials: 256 pairs over 16 moduli below 2^55.
        {"name": "batch_polymul_32768", "kind": "batch_polymul", "logn": 15, "limbs": 16,
         "polys": 256, "bits": 55},
        # Rescaling of ciphertexts in NTT form by their last modulus (64
        # polynomials of 8 limbs), the step after every product.
        {"name": "batch_rescale_65536", "kind": "batch_rescale", "logn": 16, "limbs": 8,
         "polys": 64, "bits": 50},
        # A queue of unlike jobs (transforms, products, sums; n from 2^10
        # to 2^17; 1 to 24 limbs below 2^60) as one batch.
        {"name": "mix_250", "kind": "mix", "jobs": 250, "mix_seed": 20261202},
        # The same kind of jobs arriving together at the serving engine.
        {"name": "serve_burst_64", "kind": "serve", "jobs": 64, "mix_seed": 7},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["call_polymul", "call_ntt", "call_pointwise", "batch_ntt", "batch_ntt",
                       "batch_polymul", "batch_rescale", "mix", "serve"])
    bits = rng.randint(30, 61)
    if kind == "call_polymul":
        return {"kind": kind, "logn": rng.randint(10, 17), "bits": bits}
    if kind == "call_ntt":
        return {"kind": kind, "logn": rng.randint(10, 20), "bits": bits}
    if kind == "call_pointwise":
        return {"kind": kind, "words": _log_uniform(rng, 1000, 1 << 27), "bits": bits}
    if kind in ("mix", "serve"):
        return {"kind": kind, "jobs": _log_uniform(rng, 16, 250 if kind == "mix" else 96),
                "mix_seed": rng.randrange(1 << 30)}
    logn = rng.randint(10, 20 if kind == "batch_ntt" else 17)
    limbs = rng.randint(2, 24)
    top = 1 << (25 if kind == "batch_polymul" else 26)
    polys = _log_uniform(rng, 1, max(1, top // (limbs << logn)))
    return {"kind": kind, "logn": logn, "limbs": limbs, "polys": polys, "bits": bits}


# ------------------------------------------------- moduli, tables, vectors

def _is_prime(n):
    for p in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37):
        if n % p == 0:
            return n == p
    d, s = n - 1, 0
    while d % 2 == 0:
        d, s = d // 2, s + 1
    for a in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37):
        x = pow(a, d, n)
        if x in (1, n - 1):
            continue
        for _ in range(s - 1):
            x = x * x % n
            if x == n - 1:
                break
        else:
            return False
    return True


@functools.lru_cache(maxsize=None)
def _primes(bits, count, m=1 << 21):
    """The `count` largest primes q < 2^bits with q = 1 mod m (m serves every
    n up to 2^20; narrower moduli than 2^30 do not occur here)."""
    if bits < 36:
        m = 1 << 18  # too few below 2^bits otherwise; serves n <= 2^17
    out, c = [], (((1 << bits) - 2) // m) * m + 1
    while len(out) < count and c > m:
        if _is_prime(c):
            out.append(c)
        c -= m
    return tuple(out)


@functools.lru_cache(maxsize=None)
def _root(q, n):
    """A primitive 2n-th root of unity mod q: x^((q-1)/2n) for the smallest x
    that is no square mod q."""
    x = 2
    while pow(x, (q - 1) // 2, q) != q - 1:
        x += 1
    return pow(x, (q - 1) // (2 * n), q)


@functools.lru_cache(maxsize=None)
def _context():
    return V.Context()


@functools.lru_cache(maxsize=None)
def _table(n, q):
    """Tables are made once per (n, q) and kept, as programs do."""
    return V.NttTables.on_device(_context(), n, q, _root(q, n))


def _tables(logn, limbs, bits):
    # moduli of at least 36 bits where n is past 2^17
    bits = max(bits, 36) if logn > 17 else bits
    return [_table(1 << logn, q) for q in _primes(bits, limbs)]


class _Words:
    """What __cuda_array_interface__ hands to torch: a library vector's
    words, keeping alive the object that owns them."""

    def __init__(self, owner, vector):
        self._owner = owner
        self.__cuda_array_interface__ = {
            "shape": (vector.length,), "typestr": "<i8", "version": 2,
            "data": (vector.device_ptr(), False)}


class Handles:
    """Library objects released together, the last made first."""

    def __init__(self):
        self.made = []

    def keep(self, handle):
        self.made.append(handle)
        return handle

    def __del__(self):
        for h in reversed(self.made):
            h.close()


class State:
    """One case in hand: its vectors and handles, its call, its results.
    A result tensor keeps the handles alive, not the state."""

    def __init__(self):
        self.ctx = _context()
        self.handles = Handles()

    def vector(self, words):
        return self.handles.keep(self.ctx.vector(words, zero=False))

    def view(self, base, offset, words):
        return self.handles.keep(base.view(offset, words))

    def batch(self):
        return self.handles.keep(V.Batch(self.ctx))

    def residues(self, vector, offset, polys, limbs, n, qs, gen):
        """Fills polys x limbs x n words from `offset`, limb i below qs[i]."""
        words = polys * limbs * n
        x = torch.randint(0, 1 << 62, (polys, limbs, n), generator=gen, device="cuda")
        x %= torch.tensor(qs[:limbs], device="cuda").view(1, limbs, 1)
        self.tensor(vector)[offset:offset + words] = x.view(-1)

    def tensor(self, vector):
        return torch.as_tensor(_Words(self.handles, vector), device="cuda")


# -------------------------------------------------------------- the kinds

def _prepare_call_polymul(s, case, gen):
    n = 1 << case["logn"]
    tab = _tables(case["logn"], 1, case["bits"])[0]
    a, b, fa, fb, r = (s.vector(n) for _ in range(5))
    s.residues(a, 0, 1, 1, n, [tab.q], gen)
    s.residues(b, 0, 1, 1, n, [tab.q], gen)

    def once():
        a.forward_transform(fa, tab)
        b.forward_transform(fb, tab)
        fa.elemmul(fb, r, tab.q)
        r.inverse_transform(r, tab)
    s.once, s.results = once, [fa, fb, r]


def _prepare_call_ntt(s, case, gen):
    n = 1 << case["logn"]
    tab = _tables(case["logn"], 1, case["bits"])[0]
    a, b, fa, ib = (s.vector(n) for _ in range(4))
    s.residues(a, 0, 1, 1, n, [tab.q], gen)
    s.residues(b, 0, 1, 1, n, [tab.q], gen)

    def once():
        a.forward_transform(fa, tab)
        b.inverse_transform(ib, tab)
    s.once, s.results = once, [fa, ib]


def _prepare_call_pointwise(s, case, gen):
    words = case["words"]
    q = _primes(case["bits"], 1)[0]
    a, b = s.vector(words), s.vector(words)
    out = [s.vector(words) for _ in range(5)]
    s.residues(a, 0, 1, 1, words, [q], gen)
    s.residues(b, 0, 1, 1, words, [q], gen)

    def once():
        a.elemmul(b, out[0], q)
        a.elemfma(b, out[1], 1, q)
        a.elemmod(out[2], 65537, q)
        a.elemgtadd(out[3], q // 2, 12345)
        a.elemgtsub(out[4], q // 2, 12345, 65537)
    s.once, s.results = once, out


def _slabs(s, case, gen, count):
    """`count` input slabs and their per-polynomial views."""
    n, limbs, polys = 1 << case["logn"], case["limbs"], case["polys"]
    tabs = _tables(case["logn"], limbs, case["bits"])
    limbs = len(tabs)
    made = []
    for _ in range(count):
        v = s.vector(polys * limbs * n)
        s.residues(v, 0, polys, limbs, n, [t.q for t in tabs], gen)
        made.append([s.view(v, p * limbs * n, limbs * n) for p in range(polys)])
    return n, limbs, polys, tabs, made


def _result_slab(s, polys, words):
    v = s.vector(polys * words)
    return v, [s.view(v, p * words, words) for p in range(polys)]


def _prepare_batch_ntt(s, case, gen):
    n, limbs, polys, tabs, (a,) = _slabs(s, case, gen, 1)
    spec, specs = _result_slab(s, polys, limbs * n)
    back, backs = _result_slab(s, polys, limbs * n)
    batch = s.batch()
    for p in range(polys):
        batch.add(V.JOB_NTT_FWD, a[p], None, specs[p], tabs)
    for p in range(polys):
        # another polynomial's inverse, of words that are any residues
        batch.add(V.JOB_NTT_INV, a[p], None, backs[p], tabs)
    s.once, s.results = batch.launch, [spec, back]


def _prepare_batch_polymul(s, case, gen):
    n, limbs, polys, tabs, (a, b) = _slabs(s, case, gen, 2)
    res, views = _result_slab(s, polys, limbs * n)
    batch = s.batch()
    for p in range(polys):
        batch.add(V.JOB_POLYMUL, a[p], b[p], views[p], tabs)
    s.once, s.results = batch.launch, [res]


def _prepare_batch_rescale(s, case, gen):
    n, limbs, polys, tabs, (a,) = _slabs(s, case, gen, 1)
    res, views = _result_slab(s, polys, (limbs - 1) * n)
    batch = s.batch()
    for p in range(polys):
        batch.add_rns(V.JOB_RESCALE_NTT, a[p], views[p], tabs)
    s.once, s.results = batch.launch, [res]


def _mix(case):
    """(op, log2 n, limbs) of every job."""
    rng = random.Random(case["mix_seed"])
    ops = [V.JOB_NTT_FWD, V.JOB_NTT_INV, V.JOB_POLYMUL, V.JOB_ADD_REF, V.JOB_MUL]
    return [(rng.choice(ops), rng.randint(10, 17), rng.randint(1, 24))
            for _ in range(case["jobs"])]


def _mix_jobs(s, case, gen):
    jobs = _mix(case)
    total = sum(limbs << logn for _, logn, limbs in jobs)
    qs = _primes(60, 24)
    a, b, r = (s.vector(total) for _ in range(3))
    out, at = [], 0
    for op, logn, limbs in jobs:
        n, words = 1 << logn, limbs << logn
        s.residues(a, at, 1, limbs, n, qs, gen)
        vb = None
        if op >= V.JOB_POLYMUL:
            s.residues(b, at, 1, limbs, n, qs, gen)
            vb = s.view(b, at, words)
        out.append((op, s.view(a, at, words), vb, s.view(r, at, words),
                    [_table(n, q) for q in qs[:limbs]]))
        at += words
    s.results = [r]
    return out


def _prepare_mix(s, case, gen):
    batch = s.batch()
    for job in _mix_jobs(s, case, gen):
        batch.add(*job)
    s.once = batch.launch


def _prepare_serve(s, case, gen):
    jobs = _mix_jobs(s, case, gen)
    for _, _, _, _, tabs in jobs:
        for t in tabs:
            t.upload(s.ctx)
    server = s.handles.keep(V.Server(s.ctx, scratch_bytes=1 << 28))

    def once():
        for rid in [server.submit(*job) for job in jobs]:
            status, _ = server.wait(rid)
            if status != 0:
                raise RuntimeError(f"request ended with status {status}")
    s.once = once


_PREPARE = {"call_polymul": _prepare_call_polymul, "call_ntt": _prepare_call_ntt,
            "call_pointwise": _prepare_call_pointwise, "batch_ntt": _prepare_batch_ntt,
            "batch_polymul": _prepare_batch_polymul, "batch_rescale": _prepare_batch_rescale,
            "mix": _prepare_mix, "serve": _prepare_serve}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = State()
    _PREPARE[case["kind"]](s, case, gen)
    s.outputs = [_Words(s.handles, v) for v in s.results]
    # the library works on a stream of its own: inputs are in place before it
    torch.cuda.synchronize()
    return s


def run(state):
    state.once()
    return [torch.as_tensor(w, device="cuda") for w in state.outputs]


# ------------------------------------------------------------------- work

def _ntt(words, logn):
    """Modular operations of a transform: a product, a sum and a difference
    per butterfly."""
    return 3 * words * logn // 2


def work(case):
    kind = case["kind"]
    if kind in ("mix", "serve"):
        b = f = 0
        for op, logn, limbs in _mix(case):
            words = limbs << logn
            b += 8 * words * (3 if op >= V.JOB_POLYMUL else 2)
            f += words if op > V.JOB_POLYMUL else \
                3 * _ntt(words, logn) + words if op == V.JOB_POLYMUL else _ntt(words, logn)
        return {"bytes": b, "flops": f}
    if kind == "call_pointwise":
        w = case["words"]
        return {"bytes": 8 * w * 7, "flops": 5 * w}
    logn = case["logn"]
    if kind.startswith("call"):
        w = 1 << logn
        if kind == "call_ntt":
            return {"bytes": 32 * w, "flops": 2 * _ntt(w, logn)}
        return {"bytes": 40 * w, "flops": 3 * _ntt(w, logn) + w}
    limbs, polys = case["limbs"], case["polys"]
    w = polys * limbs << logn
    if kind == "batch_ntt":
        # the one input, both results
        return {"bytes": 24 * w, "flops": 2 * _ntt(w, logn)}
    if kind == "batch_polymul":
        return {"bytes": 24 * w, "flops": 3 * _ntt(w, logn) + w}
    # rescaling: the input read, all limbs but one written
    kept = w // limbs * (limbs - 1)
    return {"bytes": 8 * (w + kept), "flops": _ntt(w, logn) + 2 * kept}


def exact(case, seed):
    """Outputs are whole numbers, the same word for word on every side."""
    return None
