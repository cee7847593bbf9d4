"""The conversions on the matrix cores (mfconv.hip) against the same context's launches through the kernel table alone
(bconv, then the transforms), word for word: one to 17 sources (padded to 8, 16 and 20, one more in the exact
conversion), targets that leave a last run of one to four, every number of targets per workgroup (1, 2, 4, 8: PCX_CC_TPW
forces the form; 0: the context's own choice of form and number), every ring degree, 28- to 31-bit primes, and ciphertexts
of words at the ends of their range (0, p - 1). Each test prints its case before the GPU runs."""
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


# (log N, Q primes, special primes, digits, bits, tops): sources of the ModUp ceil(nq / dnum), of the ModDown kp, of the
# exact conversion kp + 3
CASES = [
    (12, 3, 1, 3, 28, [2]),
    (12, 14, 8, 2, 31, [13, 6]),
    (13, 9, 5, 3, 29, [8, 3]),
    (14, 12, 4, 3, 30, [11, 10, 9]),
    (15, 18, 9, 2, 31, [17, 8]),
    (16, 20, 16, 3, 30, [19, 2]),
    (12, 34, 17, 2, 30, [33]),
    (13, 19, 18, 1, 31, [18, 5]),
]


@pytest.mark.parametrize("logn,nq,kp,dnum,bits,tops", CASES)
@pytest.mark.parametrize("tpw", [0, 1, 2, 4, 8])
def test_conversions_equal_the_tables(stream, monkeypatch, logn, nq, kp, dnum, bits, tops, tpw):
    monkeypatch.setenv("PCX_CC_TPW", str(tpw))
    ch = make("mfc", logn, nq, kp, dnum, bits)
    ctx = pa.Context(ch, k_rot=2, k_max=2)
    rng = np.random.default_rng(nq)
    s = rng.integers(-1, 2, ch.n).astype(np.int8)
    gals = [1, twin.rotation_galois(3, ch.n)]
    seeds = rng.integers(0, 2**32, (2, 8), dtype=np.uint64).astype(np.uint32)
    err = rng.integers(-3, 4, (2, ch.dnum, ch.n)).astype(np.int64)
    keys = pa.Keys(ctx, gals, seeds=seeds, secret=s, errors=err, bits=0)
    for top in tops:
        for fill in ("random", "ends"):
            ct = np.zeros((2, 2, ch.rows, ch.n), np.uint32)
            for t in range(top + 1):
                p = ch.primes[t]
                ct[:, :, t] = rng.integers(0, p, (2, 2, ch.n)) if fill == "random" else p - 1
            if fill == "ends":
                ct[:, :, :, 1::2] = 0
            x = pa.DevBuf.from_array(ct)
            out = ctx.ct_buf(2)

            def run(f):
                got = []
                for table, fused in ((False, 3), (True, 3), (False, 0)):  # the last: bconv, then whole transforms
                    ctx.table_only(table)
                    ctx.conv_fusion(fused)
                    out.zero()
                    f()
                    stream.sync()
                    got.append(out.download((2, 2, ch.rows, ch.n)))
                ctx.conv_fusion(3)
                return got

            say(f"[mfconv] N=2^{logn} {nq}+{kp} primes of {bits} bits, top {top}, {tpw} targets, {fill}: rotations")
            a, b, c = run(lambda: ctx.rotate_hoisted(keys, [0, 1], x, top, out, stream))
            for y in (b, c):
                assert (a[:, :, : top + 1] == y[:, :, : top + 1]).all()
            if top >= 2:
                say("[mfconv]   two products, rescaled (the exact conversion)")
                a, b, c = run(lambda: ctx.mul_relin_rescale(keys, x, x, top, out, stream, K=2))
                for y in (b, c):
                    assert (a[:, :, : top - 1] == y[:, :, : top - 1]).all()


def signed_digits(w, p):
    """w mod p, centred, as four signed base-256 digits (mf_digits)"""
    v = w - p if w > p // 2 else w
    d = []
    for _ in range(4):
        x = (v + 128) % 256 - 128
        d.append(x)
        v = (v - x) >> 8
    return d


@pytest.mark.parametrize("kp", [8, 16, 20])
def test_digit_sums_at_their_extremes(stream, monkeypatch, kp):
    """A ModDown whose prescaled sources are chosen against the contraction: for each target, digit and sign, coefficients
    whose bytes are 0 or 255 (in the top byte what stays below the prime) by the sign of the multiplier's digit, so that
    the digit's sum is at its most negative or positive. 31-bit primes, every padding of the sources, against the oracle"""
    monkeypatch.setenv("PCX_CC_TPW", "4")
    ch = make("ext", 12, 6, kp, 1, 31)
    ctx, oc = pa.Context(ch), twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
    top, n = len(ch.q) - 1, ch.n
    big = 1
    for p in ch.p:
        big *= int(p)
    kinds = [(t, i, sign) for t in range(top + 1) for i in range(4) for sign in (1, -1)]
    digits = {}  # [source][target][byte]: the multiplier's four digits
    for j, p in enumerate(ch.p):
        for t in range(top + 1):
            q = int(ch.q[t])
            m = big // int(p) % q
            digits[j, t] = [signed_digits(m * (1 << 8 * a) % q, q) for a in range(4)]
    ext = np.zeros((2, ch.rows, n), np.uint32)
    worst = 0
    for j, p in enumerate(ch.p):
        y = np.zeros(n, np.int64)
        for k, (t, i, sign) in enumerate(kinds):
            v = sum((255 if digits[j, t][a][i] * sign > 0 else 0) << 8 * a for a in range(4))
            y[k :: len(kinds)] = v if v < p else (v & 0xFFFFFF) | 0x7E000000
        # the INTT leaves coefficient times (P / p_j)^-1: the input's coefficients are y P / p_j
        c = (y * (big // int(p) % int(p))) % int(p)
        row = len(ch.q) + j
        ext[:, row] = oc.ntt_fwd(c.astype(np.uint32)[None].copy(), [row])[0]
    for t, i, sign in kinds:
        s = sum(abs(digits[j, t][a][i]) * (127 if digits[j, t][a][i] * sign > 0 else 128)
                for j in range(kp) for a in range(4))
        worst = max(worst, s)
    say(f"[mfconv] {kp} special primes of 31 bits: a digit's sum up to {worst} of {kp << 16}")
    assert worst > 0.3 * (kp << 16)
    rng = np.random.default_rng(kp)
    for t in range(top + 1):
        ext[:, t] = rng.integers(0, ch.primes[t], (2, n))
    dev, out = pa.DevBuf.from_array(ext), ctx.ct_buf()
    ctx.moddown(dev, top, out, stream)
    stream.sync()
    got = out.download((2, ch.rows, n))
    assert (got[:, : top + 1] == oc.moddown(ext, top)[:, : top + 1]).all()
