"""Summed rotations over `a` words expanded beforehand (kska_expand, ksum_pre_k) against the kernel table's KS_SUM dots,
which regenerate them, word for word: one, two and three digits, one and several ciphertexts, more keys than the workspace
holds at a time (the later groups added onto the first's sum), and a chain that rejects a third of the words. Each test
prints its case before the GPU runs."""
import sys

import numpy as np
import pytest

import perseus_amd as pa
from perseus_amd._lib import LIB
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


# (chain, tops, rungs' radix in bits: 2^bits - 1 keys a sum, ciphertexts)
CASES = [
    ("rej", [5, 3, 1], 4, 3),
    ((12, 7, 2, 3, 28), [6, 4, 0], 3, 5),
    ((14, 9, 4, 3, 31), [8, 5], 4, 1),
    ((16, 6, 2, 3, 30), [5, 3], 3, 6),
    ((13, 4, 1, 1, 30), [3], 2, 2),
]


@pytest.mark.parametrize("chain,tops,radix,K", CASES)
def test_sums_equal_the_tables(stream, chain, tops, radix, K):
    ch = pa.preset(chain) if chain == "rej" else make("sum", *chain)
    ctx = pa.Context(ch, k_rot=K, k_max=K)
    rng = np.random.default_rng(ch.n + K)
    s = rng.integers(-1, 2, ch.n).astype(np.int8)
    nk = (1 << radix) - 1
    gals = [twin.rotation_galois(r, ch.n) for r in range(1, nk + 1)]
    seeds = rng.integers(0, 2**32, (nk, 8), dtype=np.uint64).astype(np.uint32)
    err = rng.integers(-3, 4, (nk, ch.dnum, ch.n)).astype(np.int64)
    keys = pa.Keys(ctx, gals, seeds=seeds, secret=s, errors=err, bits=0)
    assert keys.patch_bytes() > 0
    for top in tops:
        ct = np.zeros((K, 2, ch.rows, ch.n), np.uint32)
        for t in range(top + 1):
            ct[:, :, t] = rng.integers(0, ch.primes[t], (K, 2, ch.n))
        x, out, tmp = pa.DevBuf.from_array(ct), ctx.ct_buf(K), ctx.ct_buf(K)
        say(f"[sum] {ch.name} N=2^{ch.logn} top {top}: {nk} keys, {K} ciphertexts")
        got = []
        for table in (False, True):
            ctx.table_only(table)
            out.zero()
            ctx.rotate_and_sum(keys, x, top, 1, 1 << radix, out, tmp, stream, radix_bits=radix, K=K)
            stream.sync()
            got.append(out.download((K, 2, ch.rows, ch.n))[:, :, : top + 1])
        ctx.table_only(False)
        assert (got[0] == got[1]).all()


def test_workspace(stream, monkeypatch):
    """The expanded words' workspace: none in a context without rotation keys, none with a relinearization key, three
    digits' worth of a four-digit chain with its first rotation keys; sums and a stage without it (PCX_WIDE_WS=0) and above
    three live digits equal those with it"""
    ch = make("wide", 12, 12, 2, 4, 30)
    say("[sum] four digits: the workspace, and the routes without it")
    rng = np.random.default_rng(6)
    s = rng.integers(-1, 2, ch.n).astype(np.int8)
    gals = [twin.rotation_galois(r, ch.n) for r in range(1, 4)]
    seeds = rng.integers(0, 2**32, (3, 8), dtype=np.uint64).astype(np.uint32)
    err = rng.integers(-3, 4, (3, ch.dnum, ch.n)).astype(np.int64)
    ct = np.zeros((2, ch.rows, ch.n), np.uint32)
    for t in range(len(ch.q)):
        ct[:, t] = rng.integers(0, ch.primes[t], (2, ch.n))
    x = pa.DevBuf.from_array(ct)
    pts = [pa.DevBuf.from_array(rng.integers(0, 1 << 29, (ch.rows, ch.n)).astype(np.uint32)) for _ in range(6)]
    ptrs = pa.DevBuf.from_array(np.array([p.ptr.value for p in pts], np.uint64).view(np.uint32))
    wide = 24 * ch.rows * ch.n * 4
    got = []
    for keep in ("1", "0"):
        monkeypatch.setenv("PCX_WIDE_WS", keep)
        ctx = pa.Context(ch)
        size = lambda: LIB.pcx_ctx_workspace_bytes(ctx.h)
        base = size()
        pa.Keys(ctx, [1], seeds=seeds[:1], secret=s, errors=err[:1], bits=0, relin=True)
        assert size() == base
        keys = pa.Keys(ctx, gals, seeds=seeds, secret=s, errors=err, bits=0)
        assert size() == base + (wide if keep == "1" else 0)
        res = []
        for top in (11, 8, 5):  # four, three and two live digits
            out, tmp, st = ctx.ct_buf(), ctx.ct_buf(), ctx.ct_buf(2)
            out.zero()
            st.zero()
            ctx.rotate_and_sum(keys, x, top, 1, 4, out, tmp, stream, radix_bits=2)
            ctx.cts_stage(keys, 0, 3, 2, ptrs, 6, ch.n, 0xFFFFFFFF, x, top, st, stream)
            stream.sync()
            rows = list(range(top + 1)) + [len(ch.q) + j for j in range(len(ch.p))]
            res += [out.download((2, ch.rows, ch.n))[:, : top + 1], st.download((2, 2, ch.rows, ch.n))[:, :, rows]]
        got.append(res)
    for a, b in zip(*got):
        assert (a == b).all()
