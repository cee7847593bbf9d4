"""The workloads that speed is judged by: what a program that computes on CKKS ciphertexts has this library do.

Every case goes through the package's own entry points (Rows.ntt, Context.rotate / rotate_hoisted / mul_relin /
rescale / mul_relin_rescale_list / cts_stage, attention.score_batch, bootstrap.Bootstrap.run) on ciphertexts that are
already in device memory, one context and one stream, as a serving program holds them. The shapes are the presets of
perseus_amd.chains and the benchmark's; `draw` gives others of the same ranges: ring degrees 2^12 to 2^16, 28- to 31-bit
primes, partly consumed chains (tops that leave a partial digit), any number of rotations, products or ciphertexts.

Words are residues, so every output is compared word for word. The ciphertexts' words are uniform below their primes: that
is what an encryption's words are (an encryption is indistinguishable from uniform), and no kernel's work depends on
them. Keys are made on the device from a ternary secret and rounded Gaussian errors, as key generation makes them.

A program keeps its context, its keys and its plaintext constants for its lifetime and not per ciphertext: they are made
once per shape here (`program`), and `prepare` makes the ciphertexts of a seed.
"""
import functools
import math

import torch  # first: the package then binds to the HIP runtime that torch has loaded, and one runtime serves both
import numpy as np

import perseus_amd as pa
from perseus_amd import attention, bootstrap, chains

# ---------------------------------------------------------------------------------------------------- the cases


def listed():
    c1 = dict(logn=14, nq=12, kp=4, dnum=3, bits=30)
    c3 = dict(logn=16, nq=30, kp=6, dnum=3, bits=31)
    c4 = dict(logn=16, nq=6, kp=2, dnum=3, bits=30)
    c5 = dict(logn=16, nq=47, kp=16, dnum=3, bits=30)
    return [
        # one small ciphertext into evaluation form: the smallest call, launches and latency only
        dict(name="ntt_fwd_small", op="ntt", dir=1, logn=12, polys=2, nq=6, bits=30),
        # one ciphertext of a 51-limb chain back to coefficients (before it is exported or decrypted)
        dict(name="ntt_inv_ciphertext", op="ntt", dir=-1, logn=16, polys=2, nq=51, bits=30),
        # the batched transform round trip's two directions: 64 polynomials of 40 limbs
        dict(name="ntt_fwd_batch", op="ntt", dir=1, logn=16, polys=64, nq=40, bits=31),
        dict(name="ntt_inv_batch", op="ntt", dir=-1, logn=16, polys=64, nq=40, bits=31),
        # a lone rotation on a small chain, its key bit-packed: latency
        dict(name="rotate_small", op="rotate", **c1, top=11, count=1, packed=True),
        # a lone rotation of a half-consumed ciphertext (17 limbs: the last digit is partial)
        dict(name="rotate_half_chain", op="rotate", **c3, top=16, count=1, packed=False),
        # the hoisted batch of a CoeffToSlot stage: one ModUp, 26 key switches
        dict(name="rotate_hoisted", op="rotate", **c3, top=29, count=26, packed=False),
        # one ciphertext product, relinearized, then its two-prime rescale
        dict(name="multiply", op="multiply", **c3, top=29),
        # four independent products with the rescale fused, as a polynomial evaluation takes them
        dict(name="products", op="products", **c5, top=34, count=4, packed=False),
        # encrypted attention scoring, six ciphertexts of a key cache: plaintext product, rescale, rotate-and-sum
        dict(name="scoring", op="scoring", **c4, count=6),
        # one linear-transform stage: 8 baby rotations, 8 giant steps of 63 full diagonals, in the extended basis
        dict(name="transform_stage", op="stage", **c3, top=29, babies=8, giants=8, diagonals=63),
        # the whole full-slot bootstrap, 1 limb in, 13 out
        dict(name="bootstrap", op="bootstrap", **c5),
    ]


def _chain(rng, lo, hi, logn):
    """a chain of lo..hi limbs: digits no wider than 16 limbs, every digit live, special primes near a digit's width"""
    nq = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    dnum = rng.choice([d for d in (2, 3) if nq >= d and -(-nq // d) <= 16 and -(-nq // -(-nq // d)) == d])
    alpha = -(-nq // dnum)
    kp = min(16, max(1, rng.randint((alpha + 1) // 2, alpha)))
    return dict(logn=logn, nq=nq, kp=kp, dnum=dnum, bits=rng.randint(28, 31))


def draw(rng):
    op = rng.choice(["ntt", "ntt", "rotate", "rotate", "multiply", "products", "scoring", "stage", "bootstrap"])
    logn = rng.randint(12, 16)
    if op == "ntt":
        rows = math.exp(rng.uniform(math.log(2), math.log(2560)))
        nq = min(40, max(1, round(rows ** rng.uniform(0.3, 0.9))))
        return dict(op=op, dir=rng.choice([1, -1]), logn=logn, polys=max(1, round(rows / nq)), nq=nq,
                    bits=rng.randint(28, 31))
    if op == "bootstrap":
        # the shortest chain that leaves a limb, up to 12 limbs left
        nq = rng.randint(35, 47)
        return dict(op=op, logn=rng.randint(12, 14), nq=nq, kp=-(-nq // 3), dnum=3, bits=30)
    c = _chain(rng, 4, 47 if op == "products" else 36, logn)
    # a fresh ciphertext or one with part of its chain consumed
    top = c["nq"] - 1 if rng.random() < 0.4 else rng.randint(3, c["nq"] - 1)
    if op == "rotate":
        count = round(math.exp(rng.uniform(0, math.log(26))))
        return dict(op=op, **c, top=top, count=count, packed=rng.random() < 0.3)
    if op == "multiply":
        return dict(op=op, **c, top=top)
    if op == "products":
        return dict(op=op, **c, top=top, count=rng.randint(2, 8), packed=rng.random() < 0.3)
    if op == "scoring":
        return dict(op=op, **_chain(rng, 4, 12, logn), count=rng.randint(2, 6))
    babies, giants = rng.randint(2, 8), rng.randint(1, 8)
    return dict(op=op, **c, top=top, babies=babies, giants=giants,
                diagonals=rng.randint(babies * (giants - 1) + 1, babies * giants))


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------------------------------- device words


class _Words:
    def __init__(self, ptr, words, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (words,), "typestr": "<i4", "data": (ptr, False), "version": 2}


def words(buf, offset=0, count=None):
    """the u32 words of a device buffer as a torch tensor over the same memory (int32: every word is below 2^31)"""
    count = buf.words - offset if count is None else count
    return torch.as_tensor(_Words(buf.addr(offset).value, count, buf), device="cuda")


def uniform(view, primes, gen):
    """view [..., rows, N] filled with uniform residues of row i's prime, row by row"""
    for i, p in enumerate(primes):
        shape = view.select(-2, i).shape
        view.select(-2, i).copy_(torch.randint(0, int(p), shape, generator=gen, device="cuda", dtype=torch.int32))


@functools.lru_cache(maxsize=None)
def stream():
    return pa.Stream()


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


# ---------------------------------------------------------------------------------------------------- what a program keeps


class Program:
    pass


def _keys(ctx, galois, rng, secret, packed=False, relin=False):
    ch = ctx.chain
    seeds = rng.integers(0, 1 << 32, (len(galois), 8), dtype=np.uint64).astype(np.uint32)
    errors = np.rint(rng.standard_normal((len(galois), ch.dnum, ch.n), dtype=np.float32) * 3.19).astype(np.int64)
    bits = max(p.bit_length() for p in ch.primes) if packed else 0
    return pa.Keys(ctx, galois, seeds=seeds, secret=secret, errors=errors, bits=bits, relin=relin)


@functools.lru_cache(maxsize=32)
def _program(shape):
    """the context, keys and constants of one shape (the case without its name), kept as long as the program runs"""
    case = dict(shape)
    op, P = case["op"], Program()
    logn, nq = case["logn"], case["nq"]
    n = 1 << logn
    ch = chains.make("case", logn, nq, case.get("kp", 1), case.get("dnum", 1), case["bits"])
    rng = np.random.default_rng(logn * 1000 + nq)
    secret = rng.integers(-1, 2, n).astype(np.int8)
    rot = lambda r: pow(5, r, 2 * n)
    P.chain, P.stream, count = ch, stream(), case.get("count", 1)
    if op == "ntt":
        P.ctx = pa.Context(ch)
        polys = case["polys"]
        P.rows = pa.Rows(P.ctx, list(range(polys * nq)), list(range(nq)) * polys)
    elif op == "rotate":
        # the steps of a baby-step set: 1 .. 16, then powers of two
        steps = (list(range(1, 17)) + [1 << k for k in range(5, 15)])[:count]
        P.ctx = pa.Context(ch, k_rot=count)
        P.keys = _keys(P.ctx, [rot(r) for r in steps], rng, secret, case["packed"])
    elif op == "multiply":
        P.ctx = pa.Context(ch)
        P.relin = _keys(P.ctx, [1], rng, secret, relin=True)
    elif op == "products":
        P.ctx = pa.Context(ch, k_rot=count, k_max=count)
        P.relin = _keys(P.ctx, [1], rng, secret, case["packed"], relin=True)
    elif op == "scoring":
        P.ctx = pa.Context(ch, k_rot=count, k_max=count)
        P.keys = _keys(P.ctx, [rot(r) for r in attention.ladder_steps()], rng, secret)
    elif op == "stage":
        P.ctx = pa.Context(ch)
        P.keys = _keys(P.ctx, [rot(r) for r in range(1, case["babies"])], rng, secret)
        nr = case["top"] + 1 + case["kp"]
        P.diagonals = [pa.DevBuf(nr * n) for _ in range(case["diagonals"])]
        for i, b in enumerate(P.diagonals):
            uniform(words(b).view(nr, n), ch.q[: case["top"] + 1] + ch.p, generator(i))
        P.table = pa.DevBuf.from_array(np.array([b.ptr.value for b in P.diagonals], np.uint64).view(np.uint32))
    else:
        par = bootstrap.Params(logn)
        galois, levels, conj = bootstrap.key_plan(bootstrap.Bootstrap(None, par, ch.q))
        P.ctx = pa.Context(ch, k_rot=8, k_max=8)
        P.keys = _keys(P.ctx, galois, rng, secret)
        P.relin = _keys(P.ctx, [1], rng, secret, relin=True)
        ops = bootstrap.GpuOps(P.ctx, P.keys, P.relin, levels, conj, P.stream)
        P.boot = bootstrap.Bootstrap(ops, par, ch.q, special=ch.p)
        P.boot.prepare()
    return P


def program(case):
    return _program(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


# ---------------------------------------------------------------------------------------------------- prepare and run


def prepare(case, seed):
    P, gen, op = program(case), generator(seed), case["op"]
    ctx, ch = P.ctx, P.chain
    n, rows = ch.n, ch.rows
    top = {"scoring": ch.rows - len(ch.p) - 1, "bootstrap": 0}.get(op, case.get("top"))
    s = {"case": case, "program": P, "top": top}

    def ciphertexts(count):
        buf = ctx.ct_buf(count)
        uniform(words(buf).view(count, 2, rows, n)[:, :, : top + 1], ch.q[: top + 1], gen)
        return buf

    def outputs(count, limbs, first=0):
        """count ciphertexts to write, and the rows that hold the result"""
        buf = ctx.ct_buf(count)
        words(buf).zero_()
        return buf, words(buf).view(count, 2, rows, n)[:, :, first:limbs]

    if op == "ntt":
        s["x"] = pa.DevBuf(case["polys"] * len(ch.q) * n)
        s["out"] = words(s["x"]).view(case["polys"], len(ch.q), n)
        uniform(s["out"], ch.q, gen)
    elif op == "rotate":
        s["x"] = ciphertexts(1)
        s["y"], s["out"] = outputs(case["count"], top + 1)
    elif op == "multiply":
        s["x"], s["z"] = ciphertexts(1), ciphertexts(1)
        s["y"], prod = outputs(1, top + 1)
        s["w"], rescaled = outputs(1, top - 1)
        s["out"] = (prod, rescaled)
    elif op == "products":
        # the operands sit wherever the program's buffers are: separate allocations
        s["x"] = [ciphertexts(1) for _ in range(case["count"])]
        s["z"] = [ciphertexts(1) for _ in range(case["count"])]
        s["y"], s["out"] = outputs(case["count"], top - 1)
    elif op == "scoring":
        s["x"] = ciphertexts(case["count"])
        s["pt"] = [pa.DevBuf(rows * n) for _ in range(case["count"])]
        for b in s["pt"]:
            uniform(words(b).view(rows, n)[: top + 1], ch.q[: top + 1], gen)
        s["y"], s["out"] = outputs(case["count"], top - 1)
        s["w"], _ = outputs(case["count"], 1)
    elif op == "stage":
        s["x"] = ciphertexts(1)
        s["y"], q = outputs(case["giants"], top + 1)
        s["out"] = (q, words(s["y"]).view(case["giants"], 2, rows, n)[:, :, len(ch.q):])
    else:
        s["x"] = ciphertexts(1)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return s


def run(s):
    case, P, top = s["case"], s["program"], s["top"]
    op, ctx, st = case["op"], P.ctx, P.stream
    if op == "ntt":
        P.rows.ntt(s["x"], case["dir"], st)
    elif op == "rotate":
        if case["count"] == 1:
            ctx.rotate(P.keys, 0, s["x"], top, s["y"], st)
        else:
            ctx.rotate_hoisted(P.keys, list(range(case["count"])), s["x"], top, s["y"], st)
    elif op == "multiply":
        ctx.mul_relin(P.relin, s["x"], s["z"], top, s["y"], st)
        ctx.rescale(s["y"], top, 2, s["w"], st)
    elif op == "products":
        ctx.mul_relin_rescale_list(P.relin, s["x"], s["z"], top, s["y"], st)
    elif op == "scoring":
        attention.score_batch(ctx, P.keys, s["x"], s["pt"], top, s["y"], s["w"], st)
    elif op == "stage":
        ctx.cts_stage(P.keys, 0, case["babies"], case["giants"], P.table, case["diagonals"], P.chain.n, 0xFFFFFFFF,
                      s["x"], top, s["y"], st)
    else:
        out = P.boot.run(bootstrap.View(s["x"]))
        h = words(out.h.buf, out.h.off, ctx.ct_words).view(2, ctx.rows, ctx.n)
        return h[:, : out.top + 1]
    return s["out"]


# ---------------------------------------------------------------------------------------------------- the work of a pass


@functools.lru_cache(maxsize=None)
def _stages(logn):
    cts, stc, _ = bootstrap.lt_plans(1 << logn, bootstrap.Params(logn).budget)
    shape = lambda p: (p.B, p.G, sum(v is not None for r in p.pts for v in r))
    return [shape(p) for p in cts], [shape(p) for p in stc]


def work(case):
    """the bytes of one pass: inputs, keys (their stored half) and constants read once, results written once, in rows of
    N words. The arithmetic is modular integer arithmetic and no floating-point work"""
    op, N = case["op"], 1 << case["logn"]
    if op == "ntt":
        return {"bytes": 2 * case["polys"] * case["nq"] * 4 * N}
    nq, kp = case["nq"], case["kp"]
    alpha = -(-nq // case["dnum"])
    beta = case["bits"] / 32 if case.get("packed") else 1.0
    key = lambda top: beta * (-(-(top + 1) // alpha)) * (top + 1 + kp)
    top = case.get("top", nq - 1)
    L, K = top + 1, case.get("count", 1)
    if op == "rotate":
        rows = 2 * L + K * (key(top) + 2 * L)
    elif op == "multiply":
        rows = 4 * L + key(top) + 2 * L + 2 * (L - 2)
    elif op == "products":
        rows = 4 * L * K + key(top) + 2 * (L - 2) * K
    elif op == "scoring":
        rows = K * (2 * L + L) + len(attention.ladder_steps()) * key(top - 2) + K * 2 * (L - 2)
    elif op == "stage":
        rows = 2 * L + (case["babies"] - 1) * key(top) + (case["diagonals"] + 2 * case["giants"]) * (L + kp)
    else:
        # every stage's rotation keys and diagonals (a stage's diagonals repeat every 2^s words, s the layers before it
        # on the way in and after it on the way out), and the relinearization key once per level of the sine
        cts, stc = _stages(case["logn"])
        layers = lambda st: (st[2] + 1).bit_length() - 2
        shifts = [sum(layers(x) for x in cts[:i]) for i in range(len(cts))]
        shifts += [sum(layers(x) for x in stc[i + 1:]) for i in range(len(stc))]
        rows, t, sine = 2.0 * nq, nq - 1, 7 + bootstrap.Params(case["logn"]).r
        for i, (st, s) in enumerate(zip(cts + stc, shifts)):
            if i == len(cts):
                for _ in range(sine):
                    rows += key(t)
                    t -= 2
            rows += (st[0] + st[1] - 2) * key(t) + st[2] * (t + 1 + kp) / (1 << min(s, 12))
            t -= 2
        rows += 2 * (t + 1)
    return {"bytes": rows * 4 * N}
