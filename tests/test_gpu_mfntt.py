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
from perseus_amd.chains import make
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
# rows of primes below 2^30 and of many of N = 2^15, the forward of N = 2^15 past the last-level cache
@pytest.mark.parametrize("logn,bits,rows", [
    (14, 28, 40), (14, 30, 41), (15, 28, 256), (15, 30, 257), (16, 28, 16), (16, 30, 17),
    (15, 30, 671), (15, 28, 672), (15, 31, 783), (15, 31, 784), (15, 28, 2080), (15, 30, 2081),
])
def test_transforms_at_the_rule(stream, logn, bits, rows):
    transforms(stream, logn, bits, rows)


@pytest.mark.parametrize("bits,rows", [(31, 128), (28, 129), (31, 256), (28, 257), (31, 320), (28, 321), (31, 517)])
def test_transforms_one_pass(stream, bits, rows):
    """N = 2^14 on both sides of the row counts that take one launch (N = 2^12 and 2^13 always do)"""
    transforms(stream, 14, bits, rows)


@pytest.mark.parametrize("bits,K", [(28, 4), (31, 8)])
def test_one_pass_epilogues(stream, bits, K):
    """N = 2^14 in one launch with each epilogue (the ModDown's subtraction, alone and added onto a ciphertext, the
    rescale's addition after one prime and after two, whose rows are generated), 192 to 416 rows: against the kernel table"""
    ch = make("one14", 14, 26, 7, 2, bits)
    say(f"[mfntt] N=2^14, {bits}-bit primes, {K} ciphertexts: epilogues in one launch against the kernel table")
    ctx = pa.Context(ch, k_rot=K, k_max=K)
    rng = np.random.default_rng(K)
    s = rng.integers(-1, 2, ch.n).astype(np.int8)
    gals = [twin.rotation_galois(r, ch.n) for r in (1, 2, 3)]
    seeds = rng.integers(0, 2**32, (3, 8), dtype=np.uint64).astype(np.uint32)
    err = rng.integers(-3, 4, (3, ch.dnum, ch.n)).astype(np.int64)
    keys = pa.Keys(ctx, gals, seeds=seeds, secret=s, errors=err, bits=0)
    relin = pa.Keys(ctx, [1], seeds=seeds[:1], secret=s, errors=err[:1], bits=0, relin=True)
    top, ct = 25, np.zeros((K, 2, ch.rows, ch.n), np.uint32)
    for t in range(ch.rows):
        ct[:, :, t] = rng.integers(0, ch.primes[t], (K, 2, ch.n))
    x, out, tmp = pa.DevBuf.from_array(ct), ctx.ct_buf(K), ctx.ct_buf(K)
    ctx.conv_fusion(0)  # conversions apart from the transforms, which then run whole

    def moddown():
        tmp.upload(ct, stream)  # its INTT runs in place
        ctx.moddown_k(tmp, top, out, K, stream)

    ops = [
        ("ModDown", top + 1, moddown),
        ("ModDown onto", top + 1, lambda: ctx.rotate_and_sum(keys, x, top, 1, 4, out, tmp, stream, radix_bits=2, K=K)),
        ("rescale by one", top, lambda: ctx.rescale(x, top, 1, out, stream, K=K)),
        ("rescale by two", top - 1, lambda: ctx.rescale(x, top, 2, out, stream, K=K)),
        ("product, rescaled", top - 1, lambda: ctx.mul_relin_rescale(relin, x, x, top, out, stream, K=4)),
    ]
    for name, limbs, f in ops:
        say(f"[mfntt]   {name}")
        got = []
        for table in (False, True):
            ctx.table_only(table)
            ctx.conv_fusion(0)
            out.zero()
            f()
            stream.sync()
            got.append(out.download((K, 2, ch.rows, ch.n))[:, :, :limbs])
        ctx.table_only(False)
        assert (got[0] == got[1]).all(), name


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
