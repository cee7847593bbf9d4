"""Key-switch throughput on one MI355X: the hoisted rotation batch of a CoeffToSlot BSGS stage.

Workload (the largest single-GPU configuration the metric is quoted on): one ciphertext at N = 2^16, L = 30 limbs of
31-bit primes, dnum 3 (10 limbs per digit), 6 special primes; ModUp once, then key switches to the rotation steps
{1..16, 32, 64, ..., 2^15}. 2^15 = N/2 is the identity (g = 1, a copy), so R = 26 switches. Keys: a regenerated in the
dot kernel from each key's ChaCha12 seed (the accepted redraws of its rejected words, 1-2% of them, read from a table
built with the keys and counted in the dot's bytes), b stored as dense 32-bit words (--bits 31: bit-packed, the
reference's PackedSeeded layout, 3% smaller at 31-bit primes, through the general dot); keys generated on the device
from a ternary secret (h = 192) and discrete Gaussian errors (sigma 3.19) drawn by the reference's samplers under a
fixed DRBG key (pcx_drbg_*, pcx_keygen_draw), the ciphertext uniform. One "step" = the
whole batch (ModUp + 26 dots + 26 ModDowns), inputs resident in HBM.

Prints one JSON line: value = key switches per second; roofline = the dominant stage's algorithmic bytes per launch
over its live average launch time (HIP events on its stream), with `traffic` = the HBM bytes per launch that the
FETCH_SIZE / WRITE_SIZE counters read for that kernel (profiles/traffic_c3_hoisted.json, scaled by the counters' reading
for a copy of known size); ks_roofline = the batch's algorithmic bytes over the step time; hbm_copy = the achievable
stream-copy bandwidth on this device; ntt_c2 = the batched NTT round trip (64 polynomials x 40 limbs at N = 2^16);
cpu_baseline = the oracle (this repository's C++ restatement of the reference's CPU twin) on a bounded sample of the
same batch on this host's cores.

--traffic FETCH_DIR WRITE_DIR turns two rocprofv3 --pmc runs of this script (FETCH_SIZE, then WRITE_SIZE, each also
covering the copy probe) into that traffic summary instead of benchmarking.
"""
import argparse
import math
import json
import os
import sys
import time

# the CPUs this process may use, read before any runtime starts: a runtime that binds the calling thread (an OpenMP
# or device runtime's initialisation) would make a later read report one CPU
_AFFINITY0 = sorted(os.sched_getaffinity(0))

import numpy as np  # noqa: E402

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
STEPS_SET = list(range(1, 17)) + [1 << k for k in range(5, 16)]
COPY_BYTES = 1 << 30
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "traffic_c3_hoisted.json")
# kernel of each timed stage (the rocprofv3 name prefix) and what it covers
KERNELS = {
    "dot": ("pch::ks::dot_fast<3, true, 4, 0, false>",
            "dot_fast<3, true, 4, 0, false>: key inner product of all 26 keys, a regenerated by ChaCha12"),
    "md_ntt": ("pch::ntt::mf_fwd_", "mf_fwd_rows<epilogue 1>: ModDown NTT row pass, (x - conv) P^-1"),
    "md_intt": ("pch::ntt::mf_inv_", "mf_inv_rows + mf_inv_cols: ModDown INTT of the P rows"),
    "md_bconv": ("pch::ntt::mf_conv_cols<16, 8>", "mf_conv_cols<16, 8>: ModDown P -> Q conversion and NTT column pass"),
    "modup_intt": ("pch::ntt::mf_inv_", "mf_inv_rows + mf_inv_cols: ModUp INTT"),
    "modup_bconv": ("pch::ntt::mf_conv_cols<16, 16>", "mf_conv_cols<16, 16>: ModUp conversion and NTT column pass"),
    "modup_ntt": ("pch::ntt::mf_fwd_", "mf_fwd_rows: ModUp NTT row pass"),
}


STATS_FILE = os.path.join(ROOT, "profiles", "ks_c3_hoisted_kernel_stats.md")


def rocprof_avg_us(prefix, grid=None):
    """(average us, source) of the first kernel named prefix... in the committed rocprofv3 kernel-trace summary (with
    grid: its row for that launch grid, "[grid XxYxZ]", when the summary has one), or None"""
    if not os.path.exists(STATS_FILE):
        return None
    rows = []
    for line in open(STATS_FILE):
        cells = [c.strip() for c in line.strip().strip("|").split("|")]
        if len(cells) >= 4 and cells[0].strip("`").startswith(("void " + prefix, prefix)):
            rows.append(cells)
    if grid:
        rows = [c for c in rows if f"[grid {grid}]" in c[0]] or rows
    for cells in rows:
        try:
            return float(cells[3]), os.path.relpath(STATS_FILE, ROOT)
        except ValueError:
            return None
    return None


def key_bytes_rows(ch, bits):
    """Rows of algorithmic traffic (words of N): E = D (l + k); b counted at its stored width."""
    L, k, D = len(ch.q), len(ch.p), ch.dnum
    E = D * (L + k)
    beta = (bits or 32) / 32.0
    return dict(
        E=E,
        modup=3 * E,  # INTT 2l, conversion l + (E - l), NTT 2 (E - l)
        dot=E + E * beta + L + 2 * (L + k),
        md_intt=4 * k,
        md_bconv=2 * k + 2 * L,
        md_ntt=6 * L,
        ks=E * (1 + beta) + 11 * L + 8 * k,  # one hoisted key switch (dot + ModDown)
        single=4 * E + E * beta + 11 * L + 8 * k,  # a key switch with its own ModUp
        floor=4 * L + E * beta,
    )


def host_cpu():
    """This host's CPUs: nproc, the CPUs this process may run on, one logical CPU per physical core among them (the
    reference's host pool pins one thread per physical core, crates/pc-hostrt/src/lib.rs:176-226), the model and its
    AVX-512 flags."""
    aff = _AFFINITY0
    seen, cpus = set(), []
    for c in aff:
        try:
            top = f"/sys/devices/system/cpu/cpu{c}/topology/"
            key = (open(top + "physical_package_id").read().strip(), open(top + "core_id").read().strip())
        except OSError:
            key = ("?", str(c))
        if key not in seen:
            seen.add(key)
            cpus.append(c)
    model, flags = "?", []
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name") and model == "?":
                model = line.split(":", 1)[1].strip()
            if line.startswith("flags") and not flags:
                flags = line.split(":", 1)[1].split()
    except OSError:
        pass
    return {"nproc": os.cpu_count(), "affinity_cpus": len(aff),
            "affinity_cpus_now": len(os.sched_getaffinity(0)), "physical_cores": len(cpus), "model": model,
            "avx512_flags": sorted(f for f in flags if f.startswith("avx512")), "_cpus": cpus}


def cpu_setup():
    """The oracle's pool as the reference's host runtime sizes it: min(physical cores, 36) threads, one pinned per
    physical core, and at most 16 (this GPU's share of the box's CPUs). Returns (threads, host description)."""
    from tests import twin

    h = host_cpu()
    threads = max(1, min(h["physical_cores"], 36, 16))
    twin.set_threads(threads)
    twin.set_cpus(h["_cpus"][:threads])
    desc = {k: v for k, v in h.items() if not k.startswith("_")}
    desc.update({"threads": threads, "pinned": "one thread per physical core",
                 "arithmetic": "scalar (64-bit products, 128-bit remainders); built for x86-64-v3, no AVX-512 code"})
    return threads, desc


def cpu_baseline(ch, ct, top, keys_host, gals, budget_s=10.0):
    """The oracle's hoisted batch on this host, pinned as cpu_setup() says. Cold (`a` regenerated on every call, as the
    GPU does): the sample grows to the whole batch if that fits in budget_s, then repeats until about budget_s of
    work, the rate the median over repeats. Also one thread on ModUp + 2 key switches, and the pool with the reference
    host twin's expanded-key cache warm (crates/pc-host/src/expand.rs:56-116: `a` rows kept across calls)."""
    from tests import twin

    cores, host = cpu_setup()
    oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
    seeds = np.stack([k[0] for k in keys_host])
    bs = [k[1] for k in keys_host]
    live = [i for i, g in enumerate(gals) if g != 1]

    def batch(sel):
        t0 = time.perf_counter()
        o = oc.rotate_hoisted(ct, top, seeds[sel], [bs[i] for i in sel], [gals[i] for i in sel])
        return time.perf_counter() - t0, o

    r = 2
    while True:
        sel = live[:r]
        t, outs = batch(sel)
        if r >= len(live) or t * (len(live) / r) > budget_s:
            break
        r = len(live)
    times = [t]
    while sum(times) < budget_s:
        times.append(batch(sel)[0])
    t = float(np.median(times))
    # one thread: ModUp + 2 key switches
    twin.set_threads(1)
    t1 = min(batch(live[:2])[0] for _ in range(2))
    twin.set_threads(cores)
    # the expanded-key cache warm: one call fills it, then the repeats read it
    twin.set_kska_cache(8 << 30)
    batch(sel)
    ct_times = []
    while sum(ct_times) < budget_s / 2 or len(ct_times) < 3:
        ct_times.append(batch(sel)[0])
    twin.set_kska_cache(0)
    tc = float(np.median(ct_times))
    return dict(value=r / t, unit="key-switches/s", cores=cores, kind="port",
                sample=f"ModUp + {r} hoisted key switches of the same batch (a regenerated per call, cold), median of "
                       f"{len(times)} repeats, {t:.3f} s each, {sum(times):.1f} s in all",
                single_thread={"value": round(2 / t1, 2), "unit": "key-switches/s", "threads": 1,
                               "sample": f"ModUp + 2 hoisted key switches, best of 2: {t1:.3f} s"},
                cached={"value": round(r / tc, 2), "unit": "key-switches/s", "threads": cores,
                        "sample": f"the same batch with every key's expanded a rows cached (warm), median of "
                                  f"{len(ct_times)}: {tc:.3f} s"},
                host=host), outs, sel


def hbm_copy(pa, reps=10):
    """Achievable HBM bandwidth: a plain 16-byte-access copy of COPY_BYTES, read + write counted."""
    import ctypes as C

    src, dst = pa.DevBuf(COPY_BYTES // 4), pa.DevBuf(COPY_BYTES // 4)
    st = pa.Stream()
    e0, e1 = pa.Event(), pa.Event()
    pa.check(pa.LIB.pcx_copy_probe(dst.ptr, src.ptr, C.c_size_t(COPY_BYTES), st.h), "copy_probe")
    e0.record(st)
    for _ in range(reps):
        pa.check(pa.LIB.pcx_copy_probe(dst.ptr, src.ptr, C.c_size_t(COPY_BYTES), st.h), "copy_probe")
    e1.record(st)
    st.sync()
    ms = e0.elapsed_ms(e1) / reps
    return {"bytes_copied": COPY_BYTES, "ms": round(ms, 4), "GBps": round(2 * COPY_BYTES / (ms * 1e-3) / 1e9, 1),
            "kernel": "pch::elem::copy_probe_k"}


VALU_FORMS = ("v_add_u32", "v_xor_b32", "v_alignbit_b32", "v_min_u32", "v_mul_lo_u32", "v_mul_hi_u32", "v_mad_u64_u32")


def valu_probe(pa, iters=2048, reps=3):
    """Achievable integer VALU rates: each instruction form of the kernels timed alone (pcx_valu_probe: 16 workgroups of
    256 threads per CU, 8 independent chains per thread), as wave-instructions per second, lane-operations per second
    and cycles per wave-instruction per SIMD at the device's peak clock (4 SIMDs per CU)."""
    import ctypes as C

    cus, khz = C.c_int(0), C.c_int(0)
    pa.check(pa.LIB.pc_hip_device_attribute(C.byref(cus), 16, 0), "device_attribute")
    pa.check(pa.LIB.pc_hip_device_attribute(C.byref(khz), 13, 0), "device_attribute")
    blocks = 16 * cus.value
    out = pa.DevBuf(1024)
    st = pa.Stream()
    e0, e1 = pa.Event(), pa.Event()
    forms = {}
    for kind, name in enumerate(VALU_FORMS):
        pa.check(pa.LIB.pcx_valu_probe(kind, blocks, iters, out.ptr, st.h), "valu_probe")
        e0.record(st)
        for _ in range(reps):
            pa.check(pa.LIB.pcx_valu_probe(kind, blocks, iters, out.ptr, st.h), "valu_probe")
        e1.record(st)
        st.sync()
        s = e0.elapsed_ms(e1) * 1e-3 / reps
        winstr = blocks * 4 * 8 * iters
        rate = winstr / s
        forms[name] = {"wave_instr_per_s": float(f"{rate:.4g}"), "lane_ops_T_per_s": round(rate * 64 / 1e12, 2),
                       "cycles_per_wave_instr": round(cus.value * 4 * khz.value * 1e3 / rate, 2)}
    return {"cus": cus.value, "peak_clock_mhz": khz.value // 1000, "kernel": "pch::elem::valu_probe_k",
            "note": "a wave-instruction every 4 cycles per SIMD (16 lanes) is the 39.3 T lane-ops/s of the spec's "
                    "non-packed rate; forms below 4 cycles issue faster",
            "forms": forms}


# the bench's key material: the DRBG of crates/pc-core/src/keys.rs:113-232 under a fixed key, one stream per use
KEYGEN_KEY = (0x63656E62, 0x2D68, 0x6B65, 0x7973, 2024, 0, 0, 1)


def draw_secret(pa, n):
    """the ternary secret of weight 192 (crates/pc-core/src/keys.rs:245-262) from stream 0 of the bench's DRBG"""
    return pa.Drbg(KEYGEN_KEY, 0).sparse_ternary(n, 192)


def key_draws(pa, stream, nkeys, ndig, n):
    """nkeys switching keys' seeds and Gaussian errors (sigma 3.19) from one stream of the bench's DRBG, in the order
    of the reference's key generation (pcx_keygen_draw: crates/pc-gpu/src/keygen.rs:193-210)"""
    return pa.Drbg(KEYGEN_KEY, stream).keygen_draw(nkeys, ndig, n)


def c1_leg(pa, with_cpu, reps=50):
    """The C1 workload: one rotation (r = 1) at N = 2^14, 12 limbs of 30-bit primes, dnum 3, 4 special primes, a
    ternary secret of weight 192; GPU rotations/s and, beside it, the oracle's on this host's cores (bit-exact check)."""
    ch = pa.preset("c1")
    n, top = ch.n, len(ch.q) - 1
    rng = np.random.default_rng(11)
    ctx = pa.Context(ch, k_rot=1)
    g = [pow(5, 1, 2 * n)]
    secret = draw_secret(pa, n)
    seeds, errors = key_draws(pa, 2, 1, ch.dnum, n)
    keys = pa.Keys(ctx, g, seeds=seeds, bits=30, secret=secret, errors=errors)
    ct = np.zeros((2, ch.rows, n), np.uint32)
    for part in range(2):
        for t in range(top + 1):
            ct[part, t] = rng.integers(0, ch.primes[t], n)
    st = pa.Stream()
    dev, out = pa.DevBuf.from_array(ct), ctx.ct_buf()
    for _ in range(3):
        ctx.rotate(keys, 0, dev, top, out, st)
    e0, e1 = pa.Event(), pa.Event()
    e0.record(st)
    for _ in range(reps):
        ctx.rotate(keys, 0, dev, top, out, st)
    e1.record(st)
    st.sync()
    ms = e0.elapsed_ms(e1) / reps
    res = {"workload": "one rotation, N=2^14, 12 limbs (30-bit), dnum 3, 4 special primes, packed b (30 bits)",
           "ms": round(ms, 4), "rotations_per_s": round(1e3 / ms, 1)}
    if with_cpu:
        from tests import twin

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
        b = keys.download_b(0)
        want = oc.rotate(ct, top, seeds[0], b, g[0])
        times = []
        while sum(times) < 3.0 or len(times) < 5:
            t0 = time.perf_counter()
            oc.rotate(ct, top, seeds[0], b, g[0])
            times.append(time.perf_counter() - t0)
        t = float(np.median(times))
        got = out.download((2, ch.rows, n))
        res["cpu_baseline"] = {"value": round(1.0 / t, 2), "unit": "rotations/s", "cores": cores, "kind": "port",
                               "sample": f"median of {len(times)} rotations, {t * 1e3:.1f} ms each"}
        res["cpu_gpu_bit_exact"] = bool((got[:, : top + 1] == want[:, : top + 1]).all())
    return res


def cts_leg(pa, ch, ctx, keys, seeds, ct, dev, st, with_cpu, B=8, G=8, npts=63, reps=10):
    """A CtS linear-transform stage at the C3 shape: one ModUp, then res_j = sum_{i < B} rot_i(ct) pt_{B j + i} over
    B = 8 hoisted baby rotations (steps 0..7, keys regenerated in-kernel) and G = 8 giant steps of 63 full diagonals
    (a radix-32 level of a bootstrap's CoeffToSlot), through pcx_cts_stage: the babies' dots into the context's workspace,
    then the plaintext dot over the extended rows (the timed kernel of the roofline)."""
    n, top = ch.n, len(ch.q) - 1
    nr = top + 1 + len(ch.p)
    rng = np.random.default_rng(77)
    prows = list(range(top + 1)) + [len(ch.q) + j for j in range(len(ch.p))]
    q = np.array([ch.primes[t] for t in prows], np.uint64)
    pts = [(rng.integers(0, 1 << 62, (nr, n), dtype=np.uint64) % q[:, None]).astype(np.uint32) for _ in range(npts)]
    pbufs = [pa.DevBuf.from_array(p) for p in pts]
    ptrs = pa.DevBuf.from_array(np.array([b.ptr.value for b in pbufs], np.uint64).view(np.uint32))
    res = ctx.ct_buf(G)
    for _ in range(2):
        ctx.cts_stage(keys, 0, B, G, ptrs, npts, n, 0xFFFFFFFF, dev, top, res, st)
    st.sync()
    ctx.timing(8 * reps)
    e0, e1 = pa.Event(), pa.Event()
    e0.record(st)
    for _ in range(reps):
        ctx.cts_stage(keys, 0, B, G, ptrs, npts, n, 0xFFFFFFFF, dev, top, res, st)
    e1.record(st)
    st.sync()
    ctx.timing(0)
    ms = e0.elapsed_ms(e1) / reps
    tot, cnt = ctx.timing_read()["cts"]
    launch_ms = tot / cnt
    # the plaintext dot's algorithmic rows (each operand once): the rotations, the diagonals and the results
    rows = 2 * B * nr + npts * nr + 2 * G * nr
    gbps = rows * 4 * n / (launch_ms * 1e-3) / 1e9
    out = {"workload": f"CtS stage, C3 chain at the top limb: B={B} baby rotations (a regenerated in-kernel), G={G} "
                       f"giant steps, {npts} full diagonals",
           "ms_per_stage": round(ms, 4), "stages_per_s": round(1e3 / ms, 1),
           "baby_key_switches_per_s": round((B - 1) * 1e3 / ms, 1),
           "kernel": "pt_dot_reg_k<8, 0>: the rotations times the diagonals, summed per giant step",
           "kernel_ms_per_launch": round(launch_ms, 4),
           "roofline": {"bound": "hbm", "achieved": round(gbps, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                        "frac": round(gbps / HBM_PEAK_GBPS, 4), "algorithmic_bytes_per_launch": int(rows * 4 * n)}}
    if with_cpu:
        from tests import twin

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
        bs = [keys.download_b(i) for i in range(B - 1)]
        gals = [keys.galois[i] for i in range(B - 1)]
        digits = oc.modup(ct[1], top)
        times, want = [], None
        while sum(times) < 8.0 and len(times) < 5:
            t0 = time.perf_counter()
            want = oc.cts_fused(ct[None], digits[None], top, B, G, pts, gals, seeds=seeds[: B - 1], bs=bs)[0]
            times.append(time.perf_counter() - t0)
        t = float(np.median(times))
        got = res.download((G, 2, ch.rows, n))
        out["cpu_baseline"] = {"value": round(1.0 / t, 3), "unit": "stages/s", "cores": cores, "kind": "port",
                               "sample": f"median of {len(times)} whole stages (ModUp digits precomputed), "
                                         f"{t * 1e3:.0f} ms each"}
        out["cpu_gpu_bit_exact"] = bool((got[:, :, prows] == want[:, :, prows]).all())
    return out


def mult_leg(pa, ch, ctx, secret, st, with_cpu, reps=20):
    """A relinearized product and the two-prime rescale after it at the C3 chain's top (L = 30 limbs, 31-bit primes):
    pcx_mul_relin (tensor, ModUp of d2, the relinearization key's dot with a regenerated in-kernel, ModDown added onto
    the product) then pcx_rescale (rescale_fwd: the corrections generated inside the forward NTT). The relinearization
    key is generated on the device from the batch's secret."""
    n, top = ch.n, len(ch.q) - 1
    L = top + 1
    rng = np.random.default_rng(31)
    seed, errs = key_draws(pa, 3, 1, ch.dnum, n)
    rk = pa.Keys(ctx, [1], seeds=seed, secret=secret, errors=errs, relin=True)
    host = []
    for _ in range(2):
        x = np.zeros((2, ch.rows, n), np.uint32)
        for t in range(L):
            x[:, t] = rng.integers(0, ch.primes[t], (2, n))
        host.append(x)
    da, db = pa.DevBuf.from_array(host[0]), pa.DevBuf.from_array(host[1])
    prod, rsd = ctx.ct_buf(1), ctx.ct_buf(1)
    for _ in range(2):
        ctx.mul_relin(rk, da, db, top, prod, st)
        ctx.rescale(prod, top, 2, rsd, st)
    st.sync()
    e = [pa.Event() for _ in range(4)]
    ctx.timing(16 * reps)
    e[0].record(st)
    for _ in range(reps):
        ctx.mul_relin(rk, da, db, top, prod, st)
    e[1].record(st)
    st.sync()
    ctx.timing(0)
    stages = {k: round(v[0] / reps, 4) for k, v in ctx.timing_read().items() if v[1]}
    e[2].record(st)
    for _ in range(reps):
        ctx.rescale(prod, top, 2, rsd, st)
    e[3].record(st)
    st.sync()
    mult_ms, rs_ms = e[0].elapsed_ms(e[1]) / reps, e[2].elapsed_ms(e[3]) / reps
    rows = key_bytes_rows(ch, 0)
    # algorithmic rows: the tensor reads both operands and writes (c0, c1, d2); the key switch of d2 (ModUp, dot,
    # ModDown) reads (c0, c1) once more for the add; the rescale reads the product and writes the rescaled rows
    mult_rows = 7 * L + rows["single"] + 2 * L
    rs_rows = 2 * L + 2 * (L - 2)
    mg, rg = mult_rows * 4 * n / (mult_ms * 1e-3) / 1e9, rs_rows * 4 * n / (rs_ms * 1e-3) / 1e9
    out = {"workload": f"relinearized product then a two-prime rescale, C3 chain at the top limb (L = {L})",
           "mult_ms": round(mult_ms, 4), "mults_per_s": round(1e3 / mult_ms, 1),
           "mult_stage_ms": stages,
           "rescale_ms": round(rs_ms, 4), "rescales_per_s": round(1e3 / rs_ms, 1),
           "mult_roofline": {"bound": "hbm", "achieved": round(mg, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                             "frac": round(mg / HBM_PEAK_GBPS, 4), "algorithmic_bytes": int(mult_rows * 4 * n)},
           "rescale_roofline": {"bound": "hbm", "achieved": round(rg, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                                "frac": round(rg / HBM_PEAK_GBPS, 4), "algorithmic_bytes": int(rs_rows * 4 * n)}}
    if with_cpu:
        from tests import twin

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
        bkey = rk.download_b(0)
        times, want = [], None
        while sum(times) < 6.0 and len(times) < 5:
            t0 = time.perf_counter()
            want = oc.mul_relin(host[0], host[1], top, seed[0], bkey)
            times.append(time.perf_counter() - t0)
        t = float(np.median(times))
        t0 = time.perf_counter()
        want_rs = oc.rescale(want, top, 2)
        trs = time.perf_counter() - t0
        out["cpu_baseline"] = {"value": round(1.0 / t, 3), "unit": "mults/s", "cores": cores, "kind": "port",
                               "sample": f"median of {len(times)} whole relinearized products, {t * 1e3:.0f} ms each; "
                                         f"one rescale {trs * 1e3:.0f} ms"}
        got, got_rs = prod.download((2, ch.rows, n)), rsd.download((2, ch.rows, n))
        out["cpu_gpu_bit_exact"] = bool((got[:, :L] == want[:, :L]).all() and
                                        (got_rs[:, : L - 2] == want_rs[:, : L - 2]).all())
    return out


def attn_leg(pa, secret, with_cpu, reps=10):
    """Encrypted attention scoring at the C4 shape: GPT-2-small decode, 12 heads x 64, a KV cache of 512 tokens as 6
    ciphertexts at N = 2^16 (complex packing, scale 2^40, 6 x 30-bit limbs, dnum 3, 2 special primes), the query a
    plaintext at the scale of the two primes the rescale drops. One scoring = per ciphertext a plaintext product, a
    two-prime rescale and the rotate-and-sum ladder over the 64-slot head blocks at radix 8 (two rungs of seven
    rotations hoisted over one ModUp each): 84 key switches, 12 ModUps. The keys and ciphertexts are made on the
    device (keygen, the table's encrypt from the same ternary secret). The ladders of radix 2, 4 and 64 are timed
    beside it."""
    from perseus_amd import abi, attention, encoding

    ch = pa.preset("c4")
    n, top = ch.n, len(ch.q) - 1
    ctx = pa.Context(ch, k_rot=1)
    st = pa.Stream()
    rng = np.random.default_rng(404)
    RB = attention.RADIX_BITS
    gals = [pow(5, r, 2 * n) for r in attention.ladder_steps(RB)]
    seeds, errs = key_draws(pa, 4, len(gals), ch.dnum, n)
    keys = pa.Keys(ctx, gals, seeds=seeds, secret=secret, errors=errs)
    rows = list(range(top + 1))
    ntt_rows = pa.Rows(ctx, rows, rows)
    sv = secret.astype(np.int64)
    sbuf = pa.DevBuf.from_array(np.stack([np.where(sv >= 0, sv, sv + p) for p in ch.primes[: top + 1]]).astype(np.uint32))
    ntt_rows.ntt(sbuf, 1, st)
    K = rng.normal(size=(attention.TOKENS, attention.HEADS * attention.HEAD_DIM))
    q = rng.normal(size=(attention.HEADS, attention.HEAD_DIM))
    delta = 2.0 ** 40
    enc_seed = pa.DevBuf.from_array(rng.integers(0, 1 << 32, 8, dtype=np.uint64).astype(np.uint32))
    cts, pts = [], []
    for c, z in enumerate(attention.key_slots(K, n)):
        m = np.rint(encoding.encode(z, n, delta)) + pa.Drbg(KEYGEN_KEY, 20 + c).gaussian(n)
        me = pa.DevBuf.from_array(encoding.to_residues(m, ch.primes[: top + 1]))
        ntt_rows.ntt(me, 1, st)
        ct = ctx.ct_buf(1)
        a = abi.EncryptArgs()
        a.c0, a.c1, a.s, a.e = ct.ptr.value, ct.ptr.value + 4 * ch.rows * n, sbuf.ptr.value, me.ptr.value
        a.seed, a.pr, a.nonce, a.nl = enc_seed.ptr.value, pa.LIB.pcx_ctx_primes(ctx.h), c, top + 1
        assert abi.call("encrypt", a, st, ch.logn) == 0
        cts.append(ct)
    ptscale = float(ch.q[top]) * float(ch.q[top - 1])
    for z in attention.query_slots(q, n):
        pt = pa.DevBuf(ch.rows * n)
        pt.upload(encoding.to_residues(encoding.encode(z, n, ptscale), ch.primes[: top + 1]))
        ntt_rows.ntt(pt, 1, st)
        pts.append(pt)
    outs = [ctx.ct_buf(1) for _ in cts]
    tmp = ctx.ct_buf(1)

    def scoring():
        for ct, pt, out in zip(cts, pts, outs):
            attention.score(ctx, keys, ct, pt, top, out, tmp, st)

    for _ in range(2):
        scoring()
    st.sync()
    e0, e1 = pa.Event(), pa.Event()
    e0.record(st)
    for _ in range(reps):
        scoring()
    e1.record(st)
    st.sync()
    ms = e0.elapsed_ms(e1) / reps
    # the same scoring captured once into a HIP graph and replayed: the ladder's small kernels launch as one graph
    graph = pa.Graph(st, scoring)
    for _ in range(2):
        graph.launch(st)
    st.sync()
    e0.record(st)
    for _ in range(reps):
        graph.launch(st)
    e1.record(st)
    st.sync()
    gms = e0.elapsed_ms(e1) / reps
    del graph
    # the six ciphertexts' scorings side by side: one context (workspace), key group and stream per ciphertext
    lanes = [(ctx, keys, pa.Stream(), tmp)]
    for _ in range(len(cts) - 1):
        cx = pa.Context(ch, k_rot=1)
        lanes.append((cx, pa.Keys(cx, gals, seeds=seeds, secret=secret, errors=errs), pa.Stream(), cx.ct_buf(1)))
    mouts = [ctx.ct_buf(1) for _ in cts]
    for _ in range(2):
        attention.score_streams(lanes, cts, pts, top, mouts, st)
    st.sync()
    e0.record(st)
    for _ in range(reps):
        attention.score_streams(lanes, cts, pts, top, mouts, st)
    e1.record(st)
    st.sync()
    pms = e0.elapsed_ms(e1) / reps
    same = all((a.download() == b.download()).all() for a, b in zip(mouts, outs))
    # the six ciphertexts as one batch on one stream: a context with k_max = k_rot = 6 (its keys made from the same
    # seeds, secret and errors), the rescale and every rung of the ladder as K = 6 launches (one ModUp launch sequence
    # and one ModDown per rung for the six)
    from perseus_amd.bootstrap import View

    nc = len(cts)
    cb = pa.Context(ch, k_rot=nc, k_max=nc)
    kb = pa.Keys(cb, gals, seeds=seeds, secret=secret, errors=errs)
    xb, ob, tb = cb.ct_buf(nc), cb.ct_buf(nc), cb.ct_buf(nc)
    for j, c in enumerate(cts):
        xb.upload(c.download(), offset=j * cb.ct_words)
    for _ in range(2):
        attention.score_batch(cb, kb, View(xb), pts, top, View(ob), View(tb), st)
    st.sync()
    e0.record(st)
    for _ in range(reps):
        attention.score_batch(cb, kb, View(xb), pts, top, View(ob), View(tb), st)
    e1.record(st)
    st.sync()
    bms = e0.elapsed_ms(e1) / reps
    got_b = ob.download((nc, 2, ch.rows, n))
    same_b = all((got_b[j] == o.download((2, ch.rows, n))).all() for j, o in enumerate(outs))
    if not same_b:
        raise RuntimeError("the batched scoring's words differ from the one-stream scoring's")
    # the other ladders: radix 2 (six rungs of one rotation), radix 4 (three rungs of three hoisted over one ModUp),
    # radix 64 (one rung of 63)
    radix_ms = {1 << RB: round(pms, 4)}
    for rb in (1, 2, 6):
        steps_r = attention.ladder_steps(rb)
        gals_r = [pow(5, r, 2 * n) for r in steps_r]
        seeds_r, errs_r = key_draws(pa, 10 + rb, len(gals_r), ch.dnum, n)
        lanes_r = [(cx, pa.Keys(cx, gals_r, seeds=seeds_r, secret=secret, errors=errs_r), s_, t_)
                   for cx, _, s_, t_ in lanes]
        for _ in range(2):
            attention.score_streams(lanes_r, cts, pts, top, mouts, st, radix_bits=rb)
        st.sync()
        e0.record(st)
        for _ in range(reps):
            attention.score_streams(lanes_r, cts, pts, top, mouts, st, radix_bits=rb)
        e1.record(st)
        st.sync()
        radix_ms[1 << rb] = round(e0.elapsed_ms(e1) / reps, 4)
        del lanes_r
    nks = len(cts) * len(gals)
    out = {"workload": "GPT-2-small attention scoring, 12 heads x 64, 512 cached tokens in 6 ciphertexts at N = 2^16 "
                       "(complex packing, scale 2^40): plaintext product, two-prime rescale, rotate-and-sum over 64 slots",
           "ms_per_scoring": round(bms, 4), "scorings_per_s": round(1e3 / bms, 1),
           "scores_per_s": round(attention.HEADS * attention.TOKENS * 1e3 / bms, 1),
           "timing": "the six ciphertexts as one batch on one stream (K = 6 rescale and ladder rungs)",
           "ms_per_scoring_six_streams": round(pms, 4),
           "ms_per_scoring_one_stream": round(ms, 4), "ms_per_scoring_one_stream_graph": round(gms, 4),
           "streams_equal_one_stream": bool(same), "batch_equals_one_stream": bool(same_b),
           "key_switches_per_scoring": nks, "ms_per_key_switch": round(bms / nks, 4),
           "ladder_radix": 1 << RB, "modups_per_scoring": len(cts) * -(-6 // RB),
           "ms_per_scoring_by_ladder_radix": radix_ms,
           "ladders": "rungs of radix - 1 rotations hoisted over one ModUp, on the same six streams"}
    if with_cpu:
        from oracle import em
        from tests import twin
        from tests.test_oracle_ks import decrypt

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
        s_eval = oc.secret_eval(secret)
        zs, got0 = [], None
        for i, o in enumerate(outs):
            h = o.download((2, ch.rows, n))
            got0 = h if i == 0 else got0
            coef = encoding.from_residues(decrypt(oc, s_eval, h, top - 2), ch.primes[: top - 1])
            zs.append(encoding.decode(coef, n, delta))
        want = np.einsum("hd,thd->ht", q, K.reshape(attention.TOKENS, attention.HEADS, attention.HEAD_DIM))
        out["max_score_error"] = float(np.abs(attention.scores_from_slots(zs) - want).max())
        bs = [keys.download_b(i) for i in range(len(gals))]
        ct_h = [c.download((2, ch.rows, n)) for c in cts]
        pt_h = [p.download((ch.rows, n)) for p in pts]
        times, want0 = [], None
        while sum(times) < 8.0 and len(times) < 5:
            t0 = time.perf_counter()
            for i, (x, pt) in enumerate(zip(ct_h, pt_h)):
                prod = oc.ct_zeros()
                prod[:, : top + 1] = em.mul_add_n(ch.primes, [(x[None, :, : top + 1], pt)])[0]
                r = oc.rotate_and_sum(oc.rescale(prod, top, 2), top - 2, 1, attention.BLOCK, seeds, bs, gals, RB)
                want0 = r if i == 0 else want0
            times.append(time.perf_counter() - t0)
        t = float(np.median(times))
        out["cpu_baseline"] = {"value": round(1.0 / t, 3), "unit": "scorings/s", "cores": cores, "kind": "port",
                               "sample": f"median of {len(times)} whole scorings (6 ciphertexts), {t * 1e3:.0f} ms each"}
        out["cpu_gpu_bit_exact"] = bool((got0[:, : top - 1] == want0[:, : top - 1]).all())
    return out


def bts_leg(pa, secret, with_cpu, reps=3):
    """The full-slot CKKS bootstrap at the C5 shape: N = 2^16, 2^15 complex slots uniform in [-1, 1] at scale 2^25 in
    one limb; ModRaise to 47 limbs, CoeffToSlot (4 BSGS stages), EvalMod (the reference's K = 32 series: Chebyshev
    degree 59 with the (2 pi)^(-1/8) prefactor, then 3 double angles) on the real and imaginary parts, SlotToCoeff (3
    stages): 13 limbs left; the stages are the reference's collapsed-FFT factors in FIDESlib's layout. Keys and the input
    ciphertext are made on the device from the same ternary secret; the output is decrypted (on the device, CRT on the
    host) and compared with the input's message."""
    from perseus_amd import abi, encoding
    from perseus_amd import bootstrap as B

    ch = pa.preset("c5")
    n, T = ch.n, len(ch.q) - 1
    par = B.Params(ch.logn)
    t_setup = time.perf_counter()
    gal, levels, conj = B.key_plan(B.Bootstrap(None, par, ch.q))
    ctx = pa.Context(ch, k_rot=8, k_max=8)
    rng = np.random.default_rng(505)
    seeds, errs = key_draws(pa, 6, len(gal), ch.dnum, n)
    keys = pa.Keys(ctx, gal, seeds=seeds, secret=secret, errors=errs)
    rseed, rerr = key_draws(pa, 7, 1, ch.dnum, n)
    relin = pa.Keys(ctx, [1], seeds=rseed, secret=secret, errors=rerr, relin=True)
    st = pa.Stream()
    ops = B.GpuOps(ctx, keys, relin, levels, conj, st)
    # the real and imaginary parts' EvalMod chains batched: every product, rescale and sum of the two in one launch
    # sequence (K = 2), runs of up to 8 giant steps share a ModUp and the leaves landing on one top share a rescale
    # (k_max 8)
    # every level's babies in the extended basis (a ModDown per giant step instead of per baby), CtS and StC
    boot = B.Bootstrap(ops, par, ch.q, special=ch.p, fuse_stc=True)
    assert boot.pair
    boot.prepare()
    # the input: the slots encoded at scale 2^25 with a Gaussian error folded in, encrypted at limb 0 on the device
    rows = list(range(T + 1))
    sv = secret.astype(np.int64)
    sbuf = pa.DevBuf.from_array(np.stack([np.where(sv >= 0, sv, sv + p) for p in ch.primes[: T + 1]]).astype(np.uint32))
    pa.Rows(ctx, rows, rows).ntt(sbuf, 1, st)
    z = rng.uniform(-1, 1, n // 2) + 1j * rng.uniform(-1, 1, n // 2)
    m = np.rint(encoding.encode(z, n, par.delta_in)) + pa.Drbg(KEYGEN_KEY, 30).gaussian(n)
    me = pa.DevBuf.from_array(B.residues(m, ch.primes[:1]))
    pa.Rows(ctx, [0], [0]).ntt(me, 1, st)
    x = ctx.ct_buf(1)
    enc_seed = pa.DevBuf.from_array(rng.integers(0, 1 << 32, 8, dtype=np.uint64).astype(np.uint32))
    a = abi.EncryptArgs()
    a.c0, a.c1, a.s, a.e = x.ptr.value, x.ptr.value + 4 * ch.rows * n, sbuf.ptr.value, me.ptr.value
    a.seed, a.pr, a.nonce, a.nl = enc_seed.ptr.value, pa.LIB.pcx_ctx_primes(ctx.h), 0, 1
    assert abi.call("encrypt", a, st, ch.logn) == 0
    st.sync()
    setup_s = time.perf_counter() - t_setup
    xv = B.View(x)
    out = boot.run(xv)  # warm-up: fills the buffer pool and the constant cache
    st.sync()
    ctx.timing(4096)
    boot.run(xv)
    st.sync()
    ctx.timing(0)
    stages = {k: round(v[0], 3) for k, v in ctx.timing_read().items() if v[1]}
    e0, e1 = pa.Event(), pa.Event()
    t0 = time.perf_counter()
    e0.record(st)
    for _ in range(reps):
        out = boot.run(xv)
    e1.record(st)
    st.sync()
    wall = (time.perf_counter() - t0) * 1e3 / reps
    ms = e0.elapsed_ms(e1) / reps
    # the same bootstrap with the two EvalMod chains one after the other (K = 1)
    boot.pair = False
    boot.run(xv)
    st.sync()
    e0.record(st)
    for _ in range(reps):
        out = boot.run(xv)
    e1.record(st)
    st.sync()
    ms_one = e0.elapsed_ms(e1) / reps
    boot.pair = True
    # the paired bootstrap captured into one HIP graph and replayed: no host work between the launches
    out = boot.run(xv)
    st.sync()
    eager_words = out.h.buf.download((2, ch.rows, n), offset=out.h.off, words=ctx.ct_words)
    graph = pa.Graph(st, lambda: boot.run(xv))
    graph.launch(st)
    st.sync()
    e0.record(st)
    for _ in range(reps):
        graph.launch(st)
    e1.record(st)
    st.sync()
    ms_graph = e0.elapsed_ms(e1) / reps
    graph_words = out.h.buf.download((2, ch.rows, n), offset=out.h.off, words=ctx.ct_words)
    graph_exact = bool((graph_words[:, : out.top + 1] == eager_words[:, : out.top + 1]).all())
    if not graph_exact:
        raise RuntimeError("the graph replay's output differs from the eager run's")
    # decryption: c0 + c1 s on the output's limbs (host products), INTT on the device, CRT and decoding on the host
    top = out.top
    h = out.h.buf.download((2, ch.rows, n), offset=out.h.off, words=ctx.ct_words)
    s_h = sbuf.download((T + 1, n))
    qv = np.array(ch.primes[: top + 1], np.uint64)[:, None]
    d = (h[0, : top + 1].astype(np.uint64) + h[1, : top + 1].astype(np.uint64) * s_h[: top + 1] % qv) % qv
    db = pa.DevBuf.from_array(d.astype(np.uint32))
    pa.Rows(ctx, list(range(top + 1)), list(range(top + 1))).ntt(db, -1, st)
    coef = encoding.from_residues(db.download((top + 1, n)), ch.primes[: top + 1])
    got = encoding.decode(coef, n, out.scale)
    ref = encoding.decode(m, n, par.delta_in)  # the input's message, its error included
    res = {"workload": "full-slot CKKS bootstrap, N = 2^16, 2^15 complex slots at scale 2^25 in 1 limb -> 13 limbs: "
                       "ModRaise, CtS 4 BSGS stages (babies in the extended basis, a ModDown per giant step), "
                       "EvalMod (the reference's K = 32 series: Chebyshev 59 with its prefactor + 3 double angles, "
                       "real and imaginary parts), StC 3 BSGS stages (babies in the extended basis); the reference's collapsed-FFT "
                       "factors in FIDESlib's layout",
           "chain": {"Q": len(ch.q), "P": len(ch.p), "dnum": ch.dnum, "prime_bits": 30},
           "ms_per_bootstrap": round(ms_graph, 3), "bootstraps_per_s": round(1e3 / ms_graph, 2),
           "replay": "one HIP graph of the whole bootstrap, captured once, replayed reps times",
           "graph_equals_eager": graph_exact,
           "ms_per_bootstrap_eager": round(ms, 3), "host_ms_per_bootstrap_eager": round(wall, 3), "reps": reps,
           "limbs_out": top + 1, "keys": len(gal) + 1,
           "ms_per_bootstrap_unpaired": round(ms_one, 3),
           "evalmod": "the real and imaginary parts' chains batched, K = 2 ciphertexts per launch, independent "
                      "products of one round batched further (K up to 8), each split's chain of remainders summed into "
                      "one relinearization, its last remainder rescaled with it, the basis's corrections inside their "
                      "products (unpaired: one chain after the other, eager)",
           "max_error_vs_input": float(np.abs(got - ref).max()),
           "max_error_vs_plaintext": float(np.abs(got - z).max()),
           "precision_bits": round(-math.log2(float(np.abs(got - ref).max())), 2),
           "stage_ms": stages, "setup_s": round(setup_s, 1)}
    if with_cpu:
        # one whole bootstrap on the oracle (the same keys, plans and constants; the constants' encoding done first,
        # outside the timed region, as the GPU's is), its output compared word for word with the GPU's
        from tests import twin
        from tests.bts_ops import OracleOps

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, ch.p, ch.dnum)
        bs = [keys.download_b(r) for r in range(len(gal))]
        oops = OracleOps(oc, ch.q, seeds, bs, levels, conj, rseed[0], relin.download_b(0))
        oops.set_galois(gal)
        oboot = B.Bootstrap(oops, par, ch.q, special=ch.p, fuse_stc=True)
        oboot.prepare()
        xh = x.download((2, ch.rows, n))
        t0 = time.perf_counter()
        want = oboot.run((xh[None], 0))
        t_cpu = time.perf_counter() - t0
        res["cpu_baseline"] = {
            "value": round(1.0 / t_cpu, 5), "unit": "bootstraps/s", "cores": cores, "kind": "port",
            "sample": f"one whole bootstrap of this workload on the oracle (ModRaise, CtS, both EvalMod chains one "
                      f"after the other, StC; the constants encoded beforehand): {t_cpu:.1f} s"}
        wh = OracleOps.get(want.h)
        res["cpu_gpu_bit_exact"] = bool(want.top == out.top and
                                        (eager_words[:, : out.top + 1] == wh[:, : out.top + 1]).all())
        del oops, oboot, bs
    return res


def table_leg(pa, ch, gals, seeds, secret, errors, ct_dev, top, want, steps, warmup):
    """The drop-in path: the same hoisted batch issued through the kernel table alone, as crates/pc-gpu's
    rotate_hoisted issues it (crates/pc-gpu/src/rotate.rs:456-507: the table's ntt_inv, bconv, ntt_fwd for the ModUp;
    ks_dot_key per chunk of keys; ntt_inv, bconv, ntt_fwd with the (x - conv) P^-1 epilogue for the ModDown), with
    the reference's default PackedSeeded keys (b bit-packed at the widest prime's bits, a regenerated from the seed
    in the kernel; crates/pc-gpu/src/keys.rs:24-58). The same keys' values as the headline's: outputs compared word
    for word."""
    n = ch.n
    R = sum(1 for g in gals if g != 1)
    bits = max(int(p).bit_length() for p in ch.primes)
    ctx = pa.Context(ch, k_rot=R)
    ctx.table_only(True)
    keys = pa.Keys(ctx, gals, seeds=seeds, bits=bits, secret=secret, errors=errors)
    st = pa.Stream()
    outs = ctx.ct_buf(len(gals))
    idx = list(range(len(gals)))
    for _ in range(warmup):
        ctx.rotate_hoisted(keys, idx, ct_dev, top, outs, st)
    st.sync()
    ctx.timing(16 * steps)
    e0, e1 = pa.Event(), pa.Event()
    t0 = time.perf_counter()
    e0.record(st)
    for _ in range(steps):
        ctx.rotate_hoisted(keys, idx, ct_dev, top, outs, st)
    e1.record(st)
    st.sync()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    ctx.timing(0)
    stages = {k: round(v[0] / max(v[1], 1), 4) for k, v in ctx.timing_read().items() if v[1]}
    got = outs.download((len(gals), 2, ch.rows, n))
    rows = key_bytes_rows(ch, bits)
    hoist_bytes = (rows["modup"] + R * rows["ks"]) * 4 * n
    return {"workload": "the hoisted batch through the kernel table alone, PackedSeeded keys",
            "key_b_bits": bits, "key_a": "regenerated in-kernel (ChaCha12), no retry table",
            "value": round(R / (ms * 1e-3), 1), "unit": "key-switches/s", "ms_per_step": round(ms, 4),
            "device_ms_per_step": round(e0.elapsed_ms(e1) / steps, 4), "stage_ms": stages,
            "ks_roofline_frac": round(hoist_bytes / (ms * 1e-3) / (HBM_PEAK_GBPS * 1e9), 4),
            "bit_exact_vs_headline": bool((got[:, :, : top + 1] == want[:, :, : top + 1]).all())}


def ntt_c2(pa, reps=10, with_cpu=False):
    """The batched NTT round trip: 64 polynomials x 40 limbs of 31-bit primes at N = 2^16 (2560 row transforms per
    direction), forward then inverse, the round trip checked exact."""
    ch = pa.preset("c2")
    n, npoly, L = ch.n, 64, len(ch.q)
    ctx = pa.Context(pa.Chain("c2k", ch.logn, ch.q[:-1], ch.q[-1:], 1), k_rot=1)
    rng = np.random.default_rng(7)
    q = np.array(ch.q, np.uint64)
    x = (rng.integers(0, 1 << 62, (npoly, L, n), dtype=np.uint64) % q[None, :, None]).astype(np.uint32)
    buf = pa.DevBuf.from_array(x)
    rows = pa.Rows(ctx, [p * L + t for p in range(npoly) for t in range(L)], [t for _ in range(npoly) for t in range(L)])
    st = pa.Stream()
    ev = [pa.Event() for _ in range(3)]
    rows.ntt(buf, 1, st)
    rows.ntt(buf, -1, st)
    ev[0].record(st)
    for _ in range(reps):
        rows.ntt(buf, 1, st)
    ev[1].record(st)
    for _ in range(reps):
        rows.ntt(buf, -1, st)
    ev[2].record(st)
    st.sync()
    fwd, inv = ev[0].elapsed_ms(ev[1]) / reps, ev[1].elapsed_ms(ev[2]) / reps
    exact = bool((buf.download(x.shape) == x).all())
    nrows = npoly * L
    bfly = nrows * ch.logn * (n // 2)
    row_bytes = 4 * n
    cpu = None
    if with_cpu:
        # the oracle's forward + inverse on a sample of the batch (the first 2 polynomials, 80 rows), this host's cores;
        # its forward words against the GPU's
        from tests import twin

        cores, _ = cpu_setup()
        oc = twin.Ctx(ch.logn, ch.q, [], 1)
        sample = x[:2].reshape(-1, n).copy()
        ids = [t for _ in range(2) for t in range(L)]
        times = []
        while sum(times) < 3.0 or len(times) < 3:
            t0 = time.perf_counter()
            f = oc.ntt_fwd(sample.copy(), ids)
            oc.ntt_inv(f, ids)
            times.append(time.perf_counter() - t0)
        t = float(np.median(times))
        rows.ntt(buf, 1, st)
        st.sync()
        gpu_f = buf.download(x.shape)[:2].reshape(-1, n)
        cpu = {"value": round(2 * len(ids) / t, 1), "unit": "row-transforms/s", "cores": cores, "kind": "port",
               "sample": f"forward + inverse of 80 of the 2560 rows, median of {len(times)}, {t * 1e3:.1f} ms each",
               "forward_bit_exact": bool((gpu_f == oc.ntt_fwd(sample.copy(), ids)).all())}
    return {"cpu_baseline": cpu, "rows_per_direction": nrows, "fwd_ms": round(fwd, 4), "inv_ms": round(inv, 4),
            "row_transforms_per_s": round(2 * nrows / ((fwd + inv) * 1e-3), 1),
            "butterflies_per_s": round(2 * bfly / ((fwd + inv) * 1e-3), 1),
            "GBps_algorithmic": round(2 * nrows * row_bytes / (fwd * 1e-3) / 1e9, 1),
            "kernels": "two passes per direction (a column pass, then a row pass whose loads and stores move whole cache lines)",
            "round_trip_exact": exact}


def pmc_summary(d, by_grid=False):
    """Per-kernel view of a rocprofv3 --pmc run: {kernel: {"dispatches": n, counter: [median, sum]}} over every
    counter_collection.csv under d. by_grid: one entry per kernel and grid size ("kernel [grid G]"), so that one
    workload's dispatches (the 2560-row NTT passes of C2) are not mixed with other launches of the same kernel."""
    import csv
    import glob

    vals = {}
    for f in glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True):
        for r in csv.DictReader(open(f)):
            k = r["Kernel_Name"]
            if by_grid:
                k = f"{k} [grid {r.get('Grid_Size', '?')}]"
            vals.setdefault(k, {}).setdefault(r["Counter_Name"], []).append(float(r["Counter_Value"]))
    out = {}
    for k, cs in sorted(vals.items()):
        out[k] = {"dispatches": max(len(v) for v in cs.values())}
        for c, v in sorted(cs.items()):
            out[k][c] = [float(np.median(v)), float(np.sum(v))]
    return out


def trace_summary(d, by_grid=False):
    """Markdown table of a rocprofv3 --kernel-trace run (every *kernel_trace.csv under d): calls, total ms and
    average / min / max us per kernel, slowest total first. by_grid: one row per kernel and launch grid (in threads,
    "kernel [grid XxYxZ]"), so that one workload's launches are not mixed with other launches of the same kernel."""
    import csv
    import glob

    t = {}
    for f in glob.glob(os.path.join(d, "**", "*kernel_trace.csv"), recursive=True):
        for r in csv.DictReader(open(f)):
            k = r["Kernel_Name"]
            if by_grid:
                k = f"{k} [grid {r['Grid_Size_X']}x{r['Grid_Size_Y']}x{r['Grid_Size_Z']}]"
            t.setdefault(k, []).append((int(r["End_Timestamp"]) - int(r["Start_Timestamp"])) / 1e3)
    lines = ["| kernel | calls | total ms | avg us | min us | max us |", "|---|---|---|---|---|---|"]
    for k, v in sorted(t.items(), key=lambda kv: -sum(kv[1])):
        lines.append(f"| `{k}` | {len(v)} | {sum(v) / 1e3:.3f} | {sum(v) / len(v):.1f} | {min(v):.1f} | {max(v):.1f} |")
    return "\n".join(lines)


def traffic_summary(fetch_dir, write_dir):
    """HBM bytes per dispatch of each kernel from two rocprofv3 --pmc runs (FETCH_SIZE, WRITE_SIZE, in KiB), scaled by
    the counters' reading for the copy probe (which must read and write COPY_BYTES each)."""
    fetch, write = pmc_summary(fetch_dir), pmc_summary(write_dir)
    cp = [k for k in fetch if k.startswith("pch::elem::copy_probe_k")]
    if not cp or "FETCH_SIZE" not in fetch[cp[0]] or "WRITE_SIZE" not in write.get(cp[0], {}):
        raise SystemExit("no copy probe dispatch in the counter runs")
    f_scale = COPY_BYTES / (1024.0 * fetch[cp[0]]["FETCH_SIZE"][0])
    w_scale = COPY_BYTES / (1024.0 * write[cp[0]]["WRITE_SIZE"][0])
    out = {"fetch_scale": round(f_scale, 4), "write_scale": round(w_scale, 4), "kernels": {}}
    for k, v in fetch.items():
        if "FETCH_SIZE" not in v or k.startswith("__amd"):
            continue
        fb = 1024.0 * v["FETCH_SIZE"][0] * f_scale
        wb = 1024.0 * write.get(k, {}).get("WRITE_SIZE", [0.0])[0] * w_scale
        out["kernels"][k] = {"dispatches": v["dispatches"], "fetch_bytes": round(fb), "write_bytes": round(wb),
                             "traffic_bytes": round(fb + wb)}
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--bits", type=int, default=0, help="stored width of key b (0 = dense 32-bit words)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-ntt", action="store_true", help="skip the batched NTT and C1 legs")
    ap.add_argument("--no-cts", action="store_true", help="skip the CtS stage leg")
    ap.add_argument("--no-table", action="store_true", help="skip the drop-in (kernel table only) leg")
    ap.add_argument("--no-mult", action="store_true", help="skip the relinearized product / rescale leg")
    ap.add_argument("--no-attn", action="store_true", help="skip the attention scoring leg")
    ap.add_argument("--no-bts", action="store_true", help="skip the bootstrap leg")
    ap.add_argument("--prime-bits", type=int, default=31, choices=(28, 29, 30, 31),
                    help="width of the C3 chain's primes (31: the widest the 32-bit words admit)")
    ap.add_argument("--traffic", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="summarise two rocprofv3 --pmc runs (FETCH_SIZE, WRITE_SIZE) of this script and exit")
    ap.add_argument("--pmc-summary", metavar="DIR", help="per-kernel medians / sums of a rocprofv3 --pmc run, and exit")
    ap.add_argument("--trace-summary", metavar="DIR", help="per-kernel launch times of a rocprofv3 --kernel-trace run "
                    "as a markdown table, and exit")
    ap.add_argument("--by-grid", action="store_true", help="with --pmc-summary or --trace-summary: one entry per kernel "
                    "and grid size")
    ap.add_argument("--only", choices=("ks", "ntt", "bts"), help="run one workload alone (for counter runs): the "
                    "hoisted batch without its other legs, the C2 NTT round trip alone, or the bootstrap leg alone")
    args = ap.parse_args()
    if args.traffic:
        print(json.dumps(traffic_summary(*args.traffic), indent=1))
        return
    if args.pmc_summary:
        print(json.dumps(pmc_summary(args.pmc_summary, args.by_grid), indent=1))
        return
    if args.trace_summary:
        print(trace_summary(args.trace_summary, args.by_grid))
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this library has no multi-GPU path (asked for {args.gpus})", file=sys.stderr)
        sys.exit(2)
    if args.only == "ks":
        args.no_cpu = args.no_ntt = args.no_cts = args.no_table = args.no_mult = args.no_attn = args.no_bts = True

    import perseus_amd as pa

    if args.only == "ntt":
        print(json.dumps({"ntt_c2": ntt_c2(pa)}))
        return
    if args.only == "bts":
        print(json.dumps({"bts_c5": bts_leg(pa, draw_secret(pa, 1 << 16), not args.no_cpu)}))
        return

    if pa.device_count() < 1:
        print("no GPU visible", file=sys.stderr)
        sys.exit(1)
    ch = pa.preset("c3") if args.prime_bits == 31 else pa.make_chain("c3", 16, 30, 6, 3, args.prime_bits)
    n, top = ch.n, len(ch.q) - 1
    gals = [pow(5, s % (n // 2), 2 * n) for s in STEPS_SET]
    R = sum(1 for g in gals if g != 1)
    rng = np.random.default_rng(2024)
    ctx = pa.Context(ch, k_rot=R)
    # synthetic key material, drawn as the reference's key generation draws it: a ternary secret of weight 192, each
    # key's seed and its digits' Gaussian errors (sigma 3.19) from a fixed DRBG key
    secret = draw_secret(pa, n)
    seeds, errors = key_draws(pa, 1, len(gals), ch.dnum, n)
    keys = pa.Keys(ctx, gals, seeds=seeds, bits=args.bits, secret=secret, errors=errors)
    ct = np.zeros((2, ch.rows, n), np.uint32)
    for part in range(2):
        for t in range(top + 1):
            ct[part, t] = rng.integers(0, ch.primes[t], n)
    st = pa.Stream()
    dev = pa.DevBuf.from_array(ct)
    outs = ctx.ct_buf(len(gals))
    idx = list(range(len(gals)))

    for _ in range(args.warmup):
        ctx.rotate_hoisted(keys, idx, dev, top, outs, st)
    st.sync()
    pa.check(pa.LIB.pc_hip_device_sync(), "sync")
    ctx.timing(16 * args.steps)
    e0, e1 = pa.Event(), pa.Event()
    t0 = time.perf_counter()
    e0.record(st)
    for _ in range(args.steps):
        ctx.rotate_hoisted(keys, idx, dev, top, outs, st)
    e1.record(st)
    st.sync()
    pa.check(pa.LIB.pc_hip_device_sync(), "sync")
    wall = time.perf_counter() - t0
    ctx.timing(0)
    dev_ms = e0.elapsed_ms(e1) / args.steps
    ms = wall * 1e3 / args.steps
    stages = ctx.timing_read()

    rows = key_bytes_rows(ch, args.bits)
    row_bytes = 4 * n
    # the dot also reads the key group's retry-value table (dense keys: about 1-2% of b), counted whole
    patch = keys.patch_bytes()
    per_launch_rows = {"dot": R * rows["dot"] + patch / row_bytes, "md_intt": R * rows["md_intt"], "md_bconv": R * rows["md_bconv"],
                       "md_ntt": R * rows["md_ntt"], "modup_intt": 2 * len(ch.q),
                       "modup_bconv": len(ch.q) + (rows["E"] - len(ch.q)), "modup_ntt": 2 * (rows["E"] - len(ch.q))}
    stage_info = {}
    for name, (tot, cnt) in stages.items():
        if cnt:
            avg = tot / cnt
            gbps = per_launch_rows[name] * row_bytes / (avg * 1e-3) / 1e9
            stage_info[name] = {"avg_ms": round(avg, 4), "launches": cnt, "GBps": round(gbps, 1)}
    dom = max(stage_info, key=lambda k: stage_info[k]["avg_ms"] * stage_info[k]["launches"])
    achieved = stage_info[dom]["GBps"]
    traffic, traffic_src = None, None
    if dom == "dot" and os.path.exists(TRAFFIC_FILE):
        tk = json.load(open(TRAFFIC_FILE))["kernels"]
        hit = [v for k, v in tk.items() if KERNELS[dom][0] in k]
        if hit:
            traffic, traffic_src = hit[0]["traffic_bytes"], os.path.relpath(TRAFFIC_FILE, ROOT)
    alg_bytes = per_launch_rows[dom] * row_bytes
    roofline = {"bound": "hbm", "kernel": KERNELS[dom][1], "achieved": achieved, "peak": HBM_PEAK_GBPS,
                "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBPS, 4),
                "algorithmic_bytes_per_launch": alg_bytes, "traffic": traffic, "traffic_source": traffic_src}
    avg_ms = stage_info[dom]["avg_ms"]
    if traffic:
        # the HBM bytes the counters read per launch over the same live launch time: the bandwidth the kernel
        # actually draws (below the algorithmic figure when the keys share one staging of the digits and c0)
        roofline["achieved_hbm"] = round(traffic / (avg_ms * 1e-3) / 1e9, 1)
        roofline["frac_hbm"] = round(roofline["achieved_hbm"] / HBM_PEAK_GBPS, 4)
    grid = None
    if dom == "dot":
        # the batch's dot launch (ks.hip dot_patched): N / 1024 chunks of 256 threads x the key-switch rows x key groups
        nks, chunks, groups = top + 1 + len(ch.p), n // 1024, 1
        while groups < R and chunks * nks * groups < 2048:
            groups += 1
        grid = f"{chunks * 256}x{nks}x{groups}"
    prof = rocprof_avg_us(KERNELS[dom][0], grid)
    if prof:
        # the same algorithmic bytes over the committed rocprofv3 summary's average for the kernel
        roofline["rocprof_avg_us"], roofline["rocprof_source"] = prof
        roofline["frac_rocprof"] = round(alg_bytes / (prof[0] * 1e-6) / 1e9 / HBM_PEAK_GBPS, 4)
    hoist_bytes = (rows["modup"] + R * rows["ks"]) * row_bytes + patch
    ks_gbps = hoist_bytes / (ms * 1e-3) / 1e9
    value = R / (ms * 1e-3)
    out = {
        "metric": "key-switches/sec at N=2^16 (% HBM roofline)",
        "value": round(value, 1),
        "unit": "key-switches/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "device_ms_per_step": round(dev_ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u32",
        "data": "synthetic",
        "config": {"workload": "hoisted rotation batch (CoeffToSlot BSGS)", "N": n, "L": len(ch.q), "dnum": ch.dnum,
                   "special_primes": len(ch.p), "prime_bits": args.prime_bits, "rotation_steps": STEPS_SET,
                   "key_switches_per_step": R, "key_b_bits": args.bits, "key_a": "regenerated in-kernel (ChaCha12)",
                   "key_retry_table_bytes": patch},
        "roofline": roofline,
        "ks_roofline": {"bound": "hbm", "achieved": round(ks_gbps, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                        "frac": round(ks_gbps / HBM_PEAK_GBPS, 4), "algorithmic_bytes_per_step": hoist_bytes,
                        "ks_per_s_at_peak": round(R / (hoist_bytes / (HBM_PEAK_GBPS * 1e9)), 1)},
        "stages": stage_info,
        "hbm_copy": hbm_copy(pa),
        "valu_probe": valu_probe(pa),
    }
    failed = []

    def leg(name, fn, *a, **kw):
        # a leg that fails records its error in its field; the headline line is printed all the same, and the run
        # then exits non-zero
        try:
            out[name] = fn(*a, **kw)
        except Exception as e:  # noqa: BLE001
            out[name] = {"error": f"{type(e).__name__}: {e}"}
            failed.append(name)
            print(f"bench: leg {name} failed: {e!r}", file=sys.stderr, flush=True)

    if not args.no_table:
        want = outs.download((len(gals), 2, ch.rows, n))
        leg("table_path", table_leg, pa, ch, gals, seeds, secret, errors, dev, top, want, args.steps, args.warmup)
        if isinstance(out.get("table_path"), dict) and "value" in out["table_path"]:
            out["table_path"]["vs_headline"] = round(out["table_path"]["value"] / value, 4)
    if not args.no_cts:
        leg("cts_c3", cts_leg, pa, ch, ctx, keys, seeds, ct, dev, st, not args.no_cpu)
    if not args.no_mult:
        leg("mult_c3", mult_leg, pa, ch, ctx, secret, st, not args.no_cpu)
    if not args.no_attn:
        leg("attn_c4", attn_leg, pa, secret, not args.no_cpu)
    if not args.no_bts:
        leg("bts_c5", bts_leg, pa, secret, not args.no_cpu)
    if not args.no_ntt:
        leg("ntt_c2", ntt_c2, pa, with_cpu=not args.no_cpu)
        leg("c1", c1_leg, pa, not args.no_cpu)
    if not args.no_cpu:
        host_keys = [(seeds[i], keys.download_b(i)) for i in idx]
        cpu, cpu_outs, sel = cpu_baseline(ch, ct, top, host_keys, gals)
        out["cpu_baseline"] = cpu
        # the GPU outputs of the sampled keys, word for word against the oracle's
        got = outs.download((len(gals), 2, ch.rows, n))
        out["cpu_gpu_bit_exact"] = bool(all((got[i, :, : top + 1] == cpu_outs[j][:, : top + 1]).all()
                                            for j, i in enumerate(sel)))
    if failed:
        out["failed_legs"] = failed
    print(json.dumps(out), flush=True)
    if failed:
        sys.exit(3)


if __name__ == "__main__":
    main()
