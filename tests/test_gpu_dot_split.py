"""The dot of few keys (dot_split: a wave per digit, the products exchanged through LDS) against the oracle's rotations,
word for word: two and three digits, dense keys (retry table) and packed ones at 30 and 31 bits (redrawn by the wave),
a chain that rejects a third of the words both ways, up to three keys in one launch, and launches on both sides of the
sizes from which one wave takes all digits. Each test prints its case before the GPU runs."""
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


# (chain, tops, b's width)
CASES = [
    ("rej", [5, 3], 0),
    ("rej", [5, 3], 31),
    ((12, 6, 2, 3, 30), [5, 3], 0),
    ((13, 6, 2, 3, 30), [5, 2], 30),
    ((14, 4, 2, 2, 31), [3], 31),
    ((16, 3, 1, 3, 31), [2], 0),
    ((14, 20, 8, 2, 30), [19, 9], 30),  # 448 and 1344 workgroups, 288 and 864
    ((15, 14, 4, 2, 30), [13], 0),      # 576 and 1728
]


@pytest.mark.parametrize("chain,tops,bits", CASES)
@pytest.mark.parametrize("n", [1, 3])
def test_rotations(stream, chain, tops, bits, n):
    ch = pa.preset(chain) if chain == "rej" else make("split", *chain)
    ctx, oc = pa.Context(ch, k_rot=3), twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
    g = twin.Prng([8, 7, 6, 5, 4, 3, 2, 1], 0)
    s_eval = oc.secret_eval(g.sparse_ternary(ch.n, 64))
    gals = [twin.rotation_galois(r, ch.n) for r in (1, 5, 12)][:n]
    ks = [oc.rotation_key(g, s_eval, x) for x in gals]
    seeds, bs = np.stack([k[0] for k in ks]), [k[1] for k in ks]
    keys = pa.Keys(ctx, gals, seeds=seeds, b=bs, bits=bits)
    rng = np.random.default_rng(ch.n)
    for top in tops:
        say(f"[split] {ch.name} N=2^{ch.logn} top {top}, b at {bits} bits, {n} keys")
        ct = np.zeros((2, ch.rows, ch.n), np.uint32)
        for t in range(top + 1):
            ct[:, t] = rng.integers(0, ch.primes[t], (2, ch.n))
        x, out = pa.DevBuf.from_array(ct), ctx.ct_buf(n)
        ctx.rotate_hoisted(keys, list(range(n)), x, top, out, stream)
        stream.sync()
        got = out.download((n, 2, ch.rows, ch.n))
        want = oc.rotate_hoisted(ct, top, seeds, bs, gals)
        for j in range(n):
            assert (got[j, :, : top + 1] == want[j][:, : top + 1]).all(), j
