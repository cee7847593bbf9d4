"""The matrix-core transforms (mfntt.hip) that a context's own transforms take, against the oracle's, word for word:
every ring degree (each pairs another second radix: 16 and 16, 8 and 16, 8 and 8, 4 and 8, 4 and 4), 28- to 31-bit primes
(one and two final corrections) and a chain of 31-bit primes with one far smaller among them, row counts from one, and
words at the ends of their range (0, p - 1), where a digit sum that overflowed or a bound that was short by one would
show. Chains with a prime below the matrix passes' range take the butterflies: the same words. Each test prints its case
before the GPU runs."""
import sys

import numpy as np
import pytest

import perseus_amd as pa
from tests import twin

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def stream():
    assert pa.device_count() >= 1, "no GPU visible"
    return pa.Stream()


def chain(logn, bits):
    m = 2 << logn
    if bits == "mixed":  # two corrections beside 31-bit primes
        ps = twin.descending_primes(31, m, 3) + twin.descending_primes(28, m, 2)
    elif bits == "small":  # 27-bit primes: below the range, the butterflies
        ps = twin.descending_primes(27, m, 5)
    else:
        ps = twin.descending_primes(bits, m, 5)
    return pa.Chain(f"mf{logn}_{bits}", logn, ps[:-1], ps[-1:], 1)


@pytest.mark.parametrize("logn", [12, 13, 14, 15, 16])
@pytest.mark.parametrize("bits", [28, 29, 30, 31, "mixed", "small"])
def test_transforms(stream, logn, bits):
    transforms(stream, logn, bits)


# both sides of the rows from which, or up to which, the butterflies are taken (driver.cpp mf_ntt_pays): the inverse of few
# rows of primes below 2^30, N = 2^15 past the last-level cache
@pytest.mark.parametrize("logn,bits,rows", [
    (14, 28, 40), (14, 30, 41), (15, 28, 160), (15, 30, 161), (16, 28, 16), (16, 30, 17),
    (15, 30, 2047), (15, 28, 2048), (15, 31, 2112), (15, 31, 2113),
])
def test_transforms_at_the_rule(stream, logn, bits, rows):
    transforms(stream, logn, bits, rows)


def test_transforms_one_pass(stream):
    """N = 2^14 in one pass: a launch of more rows than the two passes take (N = 2^12 and 2^13 always do)"""
    transforms(stream, 14, 31, 517)


def transforms(stream, logn, bits, rows=0):
    ch = chain(logn, bits)
    n, nq = ch.n, len(ch.q)
    rows = rows or nq + 3
    twin.set_threads(16)
    say(f"[mfntt] N=2^{logn}, {bits}-bit primes, {rows} rows: forward and inverse against the oracle")
    ctx, oc = pa.Context(ch), twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
    rng = np.random.default_rng(logn)
    ids = [i % nq for i in range(rows)]
    x = np.stack([rng.integers(0, ch.primes[i], n) for i in ids]).astype(np.uint32)
    x[0] = ch.primes[0] - 1  # every word at the top of its range
    x[1] = 0
    x[2, ::2] = ch.primes[2] - 1
    x[2, 1::2] = 0
    dev = pa.DevBuf.from_array(x)
    r = pa.Rows(ctx, list(range(rows)), ids)
    r.ntt(dev, 1, stream)
    f = dev.download((rows, n), stream=stream)
    assert (f == oc.ntt_fwd(x.copy(), ids)).all(), "forward"
    dev.upload(x, stream)
    r.ntt(dev, -1, stream)
    b = dev.download((rows, n), stream=stream)
    assert (b == oc.ntt_inv(x.copy(), ids)).all(), "inverse"
