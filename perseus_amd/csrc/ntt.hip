// Negacyclic NTT / INTT over 32-bit primes for gfx950, OpenFHE order (crates/pc-kernels/kernels/args.cuh:66-107):
// the forward transform is Cooley-Tukey with bit-reversed output, out[i] = a(psi^(2 brev(i) + 1)); the inverse is
// Gentleman-Sande with N^-1 (or a per-row scale) folded into its last pass. Twiddles: fw[m + i] = psi^brev(m + i) with
// Shoup companions (crates/pc-gpu/src/context.rs:190-230).
//
// A row of N = R x C words is viewed as R rows of C contiguous words (j = r C + c). The stages whose butterflies span
// more than C words only mix words of one column (same c): the "column pass" runs them as C independent R-point
// sub-transforms; the remaining stages stay inside one C-word block: the "row pass" runs R independent C-point
// sub-transforms. The forward runs columns then rows, the inverse rows then columns; every pass is one kernel that
// reads and writes its words once.
//
// Inside a pass each thread owns 16 words of one sub-transform of S points (T = S / 16 threads per sub-transform,
// 256 threads per workgroup): 4 butterfly stages on words spaced T apart in registers ("layout A": e = tau + T j),
// one transpose through LDS, then log2(T) stages on 16 consecutive words ("layout B": e = 16 tau + j). The inverse
// runs the same two phases in the opposite order. A row-pass sub-transform lives in one wave, so its transposes need
// only a wave barrier, and it moves its words with 16-byte accesses (layout B) around one more transpose.
//
// Butterflies are lazy. When every prime of the launch is below 2^30 (NttArgs.lazy != 0) they are Harvey's: forward
// words in [0, 4p), inverse words in [0, 2p). Otherwise (primes up to 2^31, where 4p overflows a word) forward words
// stay in [0, 2p) and inverse words canonical. Either way a transform returns canonical words.
#include "fused.h"
#include "ntt_core.h"

#include <algorithm>
#include <atomic>

namespace pch {
namespace ntt {

// ------------------------------------------------------------------------------------------------ forward
// Column pass: workgroup (x, row i) takes columns [x CC, x CC + CC) of row i. GEN: the rows are rescale corrections
// generated by RsGen from R.
template <int LOGN, bool H, bool GEN = false>
__global__ void __launch_bounds__(WG) fwd_cols(NttArgs A, int row0, RescaleArgs R = {}) {
    using G = Geo<LOGN>;
    __shared__ uint32_t lds[G::COL_LDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = row_prime(A, i);
    const uint32_t p = (uint32_t)A.pr[pid].p, p2 = 2 * p;
    const uint32_t* w = (const uint32_t*)A.fw + ((size_t)pid << LOGN);
    const uint32_t* ws = (const uint32_t*)A.fws + ((size_t)pid << LOGN);
    const int col = threadIdx.x % G::CC, tau = threadIdx.x / G::CC;
    const int c = B.x * G::CC + col;
    uint32_t x[E];
    if (GEN) {
        const RsGen gen(R, (const uint32_t*)A.base + (row_off(A, i) << LOGN), pid, LOGN);
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = gen((size_t)(tau + G::TR * j) * G::C + c);
    } else {
        const RowSrc src = row_src(A, i, LOGN);
        if (src.n == 1) {
            // through a buffer resource: one per-lane offset, each word's row offset a scalar
            const Buf bs(src.p0, (uint32_t)G::N * 4);
            const uint32_t vo = (uint32_t)(tau * G::C + c) * 4;
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = bs.ld(vo, (uint32_t)(G::TR * j * G::C) * 4);
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = ld_src(src, (size_t)(tau + G::TR * j) * G::C + c, p);
        }
    }
    // stages h = R/2 .. TR (rows): index R/(2h) + r/(2h)
    auto base = [](int h) { return (uint32_t)(G::R / (2 * h)); };
    phase_a<true, H, G::TR, decltype(base), true>(x, w, ws, p, p2, base);
#pragma unroll
    for (int j = 0; j < E; ++j) lds[tau * G::WT + col + j * G::WS] = x[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = lds[tau * G::RT + col + j * G::RS];
    phase_b<true, H, G::TR>(x, tau, w, ws, p, p2, base);
    const Buf bo((const uint32_t*)A.base + (row_off(A, i) << LOGN), (uint32_t)G::N * 4);
    const uint32_t vo = (uint32_t)(E * tau * G::C + c) * 4;
#pragma unroll
    for (int j = 0; j < E; ++j) bo.st(x[j], vo, (uint32_t)(j * G::C) * 4);  // lazy words
}

// Row pass: workgroup (x, row i) takes blocks [x BB, x BB + BB) of row i (C contiguous words each). EPI: NttArgs.epi
// (0: in place; 1: eout = (x - v) s, 2: eout = d + (x - v) s, 3: eout = x s + v; x = the sum of xnum rows of ex,
// s = es[prime id]; args.cuh:66-80).
template <int LOGN, bool H, int EPI>
__global__ void __launch_bounds__(WG) fwd_rows(NttArgs A, int row0) {
    using G = Geo<LOGN>;
    __shared__ uint32_t lds[G::ROW_LDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = row_prime(A, i);
    const uint32_t p = (uint32_t)A.pr[pid].p, p2 = 2 * p;
    const uint32_t* w = (const uint32_t*)A.fw + ((size_t)pid << LOGN);
    const uint32_t* ws = (const uint32_t*)A.fws + ((size_t)pid << LOGN);
    const int lb = threadIdx.x / G::TC, tau = threadIdx.x % G::TC;
    const int blk = B.x * G::BB + lb;
    auto base = [blk](int h) { return (uint32_t)((G::N / (2 * h)) + blk * (G::C / (2 * h))); };
    if constexpr (G::C == 256) {
        // the D / E layouts: whole-line loads and stores
        const size_t r0 = (row_off(A, i) << LOGN) + (size_t)blk * G::C + 4 * tau;
        uint32_t* a = (uint32_t*)A.base + r0;
        uint32_t x[E];
        // with an epilogue the row's words are read once (the column pass's output, or a conversion's): streamed past
        // the caches
        if (EPI != 0) ld_d_nt(a, x);
        else ld_d(a, x);
        uint32_t* l = lds + lb * (G::C + G::C / E);
        stages_hi_d<true, H>(x, w, ws, base, p, p2);
        Tw te;
        load_tw_e(te, w, ws, base, tau >> 2);
        d_to_e(x, l, tau);
        phase_a_t<true, H>(x, te, p, p2);
        e_to_d(x, l, tau);
        stages_lo_d<true, H>(x, w, ws, base, tau, p, p2);
        // the epilogue's operand after the butterflies, also streamed: 78 registers instead of 99 (6 waves per SIMD
        // instead of 4), whose other waves cover the loads' latency (the C3 ModDown's row pass: 0.269 -> 0.240 ms)
        uint32_t ex[E];
        if (EPI != 0) {
            const RowSrc xs{(const uint32_t*)A.ex, A.xnum, A.xstride};
            if (xs.n == 1) ld_d_nt(xs.p0 + r0, ex);
            else ld_d_src(xs, r0, p, ex);
        }
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = canon<H>(x[j], p, p2);
        if (EPI == 0) {
            st_d(a, x);
            return;
        }
        const uint32_t s = ((const uint32_t*)A.es)[pid], ss = ((const uint32_t*)A.ess)[pid];
        uint32_t* o = (uint32_t*)A.eout + r0;
        uint32_t d[E];
        if (EPI == 2) ld_d(A.ed ? (const uint32_t*)A.ed + r0 : o, d);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            if (EPI == 3) {
                x[j] = addm(shoup(ex[j], s, ss, p), x[j], p);
            } else {
                const uint32_t y = shoup(ex[j] - x[j] + p, s, ss, p);
                x[j] = EPI == 2 ? addm(d[j], y, p) : y;
            }
        }
        st_d(o, x);
        return;
    }
    const size_t r0 = (row_off(A, i) << LOGN) + (size_t)blk * G::C + E * tau;
    uint32_t* a = (uint32_t*)A.base + r0;
    uint32_t x[E];
    ld16(a, x);
    // the epilogue's operand is loaded with the row: every HBM read of the workgroup is in flight before the butterflies
    uint32_t ex[E];
    if (EPI != 0) ld16_src(RowSrc{(const uint32_t*)A.ex, A.xnum, A.xstride}, r0, p, ex);
    constexpr int LS = G::C + G::C / E;
    uint32_t* l = lds + lb * LS;
    // stage of half distance h (words): index N/(2h) + blk C/(2h) + c/(2h)
    Tw ta, tb;
    load_tw_a<G::TC>(ta, w, ws, base);
    b_to_a<G::TC>(x, l, tau);
    phase_a_t<true, H>(x, ta, p, p2);
    // phase B's twiddles after phase A's die: fewer live registers, more waves per SIMD
    load_tw_b<G::TC>(tb, tau, w, ws, base);
    a_to_b<G::TC>(x, l, tau);
    phase_b_t<true, H, G::TC>(x, tb, p, p2);
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = canon<H>(x[j], p, p2);
    if (EPI == 0) {
        st16(a, x);
        return;
    }
    const uint32_t s = ((const uint32_t*)A.es)[pid], ss = ((const uint32_t*)A.ess)[pid];
    uint32_t* o = (uint32_t*)A.eout + r0;
    uint32_t d[E];
    if (EPI == 2) ld16(A.ed ? (const uint32_t*)A.ed + r0 : o, d);
#pragma unroll
    for (int j = 0; j < E; ++j) {
        if (EPI == 3) {
            x[j] = addm(shoup(ex[j], s, ss, p), x[j], p);
        } else {
            const uint32_t y = shoup(ex[j] - x[j] + p, s, ss, p);
            x[j] = EPI == 2 ? addm(d[j], y, p) : y;
        }
    }
    st16(o, x);
}

// ------------------------------------------------------------------------------------------------ inverse
template <int LOGN, bool H>
__global__ void __launch_bounds__(WG) inv_rows(NttArgs A, int row0) {
    using G = Geo<LOGN>;
    __shared__ uint32_t lds[G::ROW_LDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = row_prime(A, i);
    const uint32_t p = (uint32_t)A.pr[pid].p, p2 = 2 * p;
    const uint32_t* w = (const uint32_t*)A.iw + ((size_t)pid << LOGN);
    const uint32_t* ws = (const uint32_t*)A.iws + ((size_t)pid << LOGN);
    const int lb = threadIdx.x / G::TC, tau = threadIdx.x % G::TC;
    const int blk = B.x * G::BB + lb;
    const RowSrc src = row_src(A, i, LOGN);
    auto base = [blk](int h) { return (uint32_t)((G::N / (2 * h)) + blk * (G::C / (2 * h))); };
    if constexpr (G::C == 256) {
        // the D / E layouts: whole-line loads and stores
        const size_t e0 = (size_t)blk * G::C + 4 * tau;
        uint32_t x[E];
        ld_d_src(src, e0, p, x);
        uint32_t* l = lds + lb * (G::C + G::C / E);
        stages_lo_d<false, H>(x, w, ws, base, tau, p, p2);
        Tw te;
        load_tw_e(te, w, ws, base, tau >> 2);
        d_to_e(x, l, tau);
        phase_a_t<false, H>(x, te, p, p2);
        e_to_d(x, l, tau);
        stages_hi_d<false, H>(x, w, ws, base, p, p2);
        st_d((uint32_t*)A.base + (row_off(A, i) << LOGN) + e0, x);  // [0, 2p) (Harvey) or canonical
        return;
    }
    const size_t e0 = (size_t)blk * G::C + E * tau;
    uint32_t x[E];
    ld16_src(src, e0, p, x);
    Tw ta, tb;
    load_tw_b<G::TC>(tb, tau, w, ws, base);
    phase_b_t<false, H, G::TC>(x, tb, p, p2);
    load_tw_a<G::TC>(ta, w, ws, base);
    constexpr int LS = G::C + G::C / E;
    uint32_t* l = lds + lb * LS;
    b_to_a<G::TC>(x, l, tau);
    phase_a_t<false, H>(x, ta, p, p2);
    a_to_b<G::TC>(x, l, tau);
    st16((uint32_t*)A.base + (row_off(A, i) << LOGN) + e0, x);  // [0, 2p) (Harvey) or canonical
}

template <int LOGN, bool H>
__global__ void __launch_bounds__(WG) inv_cols(NttArgs A, int row0) {
    using G = Geo<LOGN>;
    __shared__ uint32_t lds[G::COL_LDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = row_prime(A, i);
    const uint32_t p = (uint32_t)A.pr[pid].p, p2 = 2 * p;
    const uint32_t* w = (const uint32_t*)A.iw + ((size_t)pid << LOGN);
    const uint32_t* ws = (const uint32_t*)A.iws + ((size_t)pid << LOGN);
    const int col = threadIdx.x % G::CC, tau = threadIdx.x / G::CC;
    const int c = B.x * G::CC + col;
    const Buf ba((const uint32_t*)A.base + (row_off(A, i) << LOGN), (uint32_t)G::N * 4);
    uint32_t x[E];
    const uint32_t vi = (uint32_t)(E * tau * G::C + c) * 4;
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = ba.ld(vi, (uint32_t)(j * G::C) * 4);
    auto base = [](int h) { return (uint32_t)(G::R / (2 * h)); };
    phase_b<false, H, G::TR>(x, tau, w, ws, p, p2, base);
#pragma unroll
    for (int j = 0; j < E; ++j) lds[tau * G::RT + col + j * G::RS] = x[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = lds[tau * G::WT + col + j * G::WS];
    phase_a<false, H, G::TR, decltype(base), true>(x, w, ws, p, p2, base);
    // the scale: es[i] per row (NttArgs ABI 17) or N^-1 of the prime; Shoup takes the lazy words whole
    uint32_t s, ss;
    if (A.es) {
        s = ((const uint32_t*)A.es)[i];
        ss = ((const uint32_t*)A.ess)[i];
    } else {
        s = ((const uint32_t*)A.ninv)[pid];
        ss = ((const uint32_t*)A.ninvs)[pid];
    }
    const uint32_t vo = (uint32_t)(tau * G::C + c) * 4;
#pragma unroll
    for (int j = 0; j < E; ++j) ba.st(shoup(x[j], s, ss, p), vo, (uint32_t)(G::TR * j * G::C) * 4);
}

// ------------------------------------------------------------------------------------------------ launchers
inline int check(const NttArgs* a, bool fwd) {
    if (!a || a->nrows < 0 || !a->base || !a->roff || !a->rprime || !a->pr) return -1;
    if (fwd ? (!a->fw || !a->fws) : (!a->iw || !a->iws)) return -1;
    if (a->soff && (!a->src || a->snum < 1)) return -1;
    if (fwd && a->epi != 0) {
        if (a->epi < 1 || a->epi > 3 || !a->eout || !a->ex || !a->es || !a->ess || a->xnum < 1) return -2;
    } else if (a->epi != 0) {
        return -2;  // the epilogues exist on the forward transform only
    }
    if (!fwd && !a->es && (!a->ninv || !a->ninvs)) return -1;
    return 0;
}

template <int LOGN, bool H, bool GEN = false>
void fwd_pair(const NttArgs& A, int r0, int n, hipStream_t st, const RescaleArgs& R = {}) {
    using G = Geo<LOGN>;
    // a first pass out of place (or generated), then the row pass in place on base
    hipLaunchKernelGGL((fwd_cols<LOGN, H, GEN>), dim3(G::COL_WGS, n), dim3(WG), 0, st, A, r0, R);
    NttArgs B = A;
    B.soff = nullptr;
    const dim3 g(G::ROW_WGS, n);
    switch (A.epi) {
        case 0: hipLaunchKernelGGL((fwd_rows<LOGN, H, 0>), g, dim3(WG), 0, st, B, r0); break;
        case 1: hipLaunchKernelGGL((fwd_rows<LOGN, H, 1>), g, dim3(WG), 0, st, B, r0); break;
        case 2: hipLaunchKernelGGL((fwd_rows<LOGN, H, 2>), g, dim3(WG), 0, st, B, r0); break;
        default: hipLaunchKernelGGL((fwd_rows<LOGN, H, 3>), g, dim3(WG), 0, st, B, r0); break;
    }
}

// Launches of at least ntt1_min() rows of N = 2^16 run the one-pass transform (ntt1.hip: one workgroup per row, each
// word through HBM once); the others the two-pass. Off by default: since the row pass moves whole cache lines, the
// two-pass is the faster on every batch measured on MI355X (2560 rows: 0.72 ms against 0.78 forward and inverse; 312
// rows: the one-pass needs two rounds of the 256 CUs). PCX_NTT1_MIN sets the threshold at the first launch,
// pcx_ntt_one_pass_min at any time (0: never).
std::atomic<int> g_ntt1_min{-1};
inline int ntt1_min() {
    int v = g_ntt1_min.load(std::memory_order_relaxed);
    if (v < 0) {
        const char* e = getenv("PCX_NTT1_MIN");
        v = e ? std::max(0, atoi(e)) : 0;
        int expect = -1;
        if (!g_ntt1_min.compare_exchange_strong(expect, v)) v = expect;
    }
    return v;
}
inline bool one_pass(int logn, int n) { return logn == 16 && ntt1_min() > 0 && n >= ntt1_min(); }

template <int LOGN>
int fwd(const NttArgs* a, pc_stream_t s) {
    if (int rc = check(a, true)) return rc;
    const NttArgs A = *a;
    const int chunk = A.chunk > 0 ? A.chunk : (A.nrows > 0 ? A.nrows : 1);
    hipStream_t st = (hipStream_t)s;
    for (int r0 = 0; r0 < A.nrows; r0 += chunk) {
        const int n = A.nrows - r0 < chunk ? A.nrows - r0 : chunk;
        // the one-pass forward reads an epilogue's operand only after its butterflies (one workgroup per CU, nothing
        // to overlap it with): the two-pass row pass, whose epilogue streams beside other workgroups' butterflies,
        // is faster there (1560 ModDown rows on MI355X: 0.61 ms one-pass against 0.48 ms two-pass)
        if (one_pass(LOGN, n) && A.epi == 0) ntt1_fwd(A, r0, n, s);
        else if (A.lazy) fwd_pair<LOGN, true>(A, r0, n, st);
        else fwd_pair<LOGN, false>(A, r0, n, st);
    }
    return launch_rc();
}

template <int LOGN, bool H>
void inv_pair(const NttArgs& A, int r0, int n, hipStream_t st) {
    using G = Geo<LOGN>;
    hipLaunchKernelGGL((inv_rows<LOGN, H>), dim3(G::ROW_WGS, n), dim3(WG), 0, st, A, r0);
    NttArgs B = A;
    B.soff = nullptr;
    hipLaunchKernelGGL((inv_cols<LOGN, H>), dim3(G::COL_WGS, n), dim3(WG), 0, st, B, r0);
}

template <int LOGN>
int inv(const NttArgs* a, pc_stream_t s) {
    if (int rc = check(a, false)) return rc;
    const NttArgs A = *a;
    const int chunk = A.chunk > 0 ? A.chunk : (A.nrows > 0 ? A.nrows : 1);
    hipStream_t st = (hipStream_t)s;
    for (int r0 = 0; r0 < A.nrows; r0 += chunk) {
        const int n = A.nrows - r0 < chunk ? A.nrows - r0 : chunk;
        if (one_pass(LOGN, n)) ntt1_inv(A, r0, n, s);
        else if (A.lazy) inv_pair<LOGN, true>(A, r0, n, st);
        else inv_pair<LOGN, false>(A, r0, n, st);
    }
    return launch_rc();
}

// the row pass alone over every row of the args (after a column pass done elsewhere)
template <int LOGN>
int fwd_rows_only(const NttArgs* a, pc_stream_t s) {
    if (int rc = check(a, true)) return rc;
    using G = Geo<LOGN>;
    if (a->nrows == 0) return 0;
    NttArgs B = *a;
    B.soff = nullptr;
    const dim3 g(G::ROW_WGS, B.nrows);
    hipStream_t st = (hipStream_t)s;
#define PCH_ROWS(HH)                                                                               \
    switch (B.epi) {                                                                               \
        case 0: hipLaunchKernelGGL((fwd_rows<LOGN, HH, 0>), g, dim3(WG), 0, st, B, 0); break;     \
        case 1: hipLaunchKernelGGL((fwd_rows<LOGN, HH, 1>), g, dim3(WG), 0, st, B, 0); break;     \
        case 2: hipLaunchKernelGGL((fwd_rows<LOGN, HH, 2>), g, dim3(WG), 0, st, B, 0); break;     \
        default: hipLaunchKernelGGL((fwd_rows<LOGN, HH, 3>), g, dim3(WG), 0, st, B, 0); break;    \
    }
    if (B.lazy) {
        PCH_ROWS(true)
    } else {
        PCH_ROWS(false)
    }
#undef PCH_ROWS
    return launch_rc();
}

// the forward transform of rescale corrections generated in the column pass (R: the rescale, ndrop 2)
template <int LOGN>
int fwd_rescale(const NttArgs* a, const RescaleArgs* R, pc_stream_t s) {
    if (int rc = check(a, true)) return rc;
    if (a->soff) return -1;
    const NttArgs A = *a;
    const int chunk = A.chunk > 0 ? A.chunk : (A.nrows > 0 ? A.nrows : 1);
    hipStream_t st = (hipStream_t)s;
    for (int r0 = 0; r0 < A.nrows; r0 += chunk) {
        const int n = A.nrows - r0 < chunk ? A.nrows - r0 : chunk;
        if (A.lazy) fwd_pair<LOGN, true, true>(A, r0, n, st, *R);
        else fwd_pair<LOGN, false, true>(A, r0, n, st, *R);
    }
    return launch_rc();
}

}  // namespace ntt

int ntt_fwd_rescale(int logn, const NttArgs* a, const RescaleArgs* r, pc_stream_t s) {
    switch (logn) {
        case 12: return ntt::fwd_rescale<12>(a, r, s);
        case 13: return ntt::fwd_rescale<13>(a, r, s);
        case 14: return ntt::fwd_rescale<14>(a, r, s);
        case 15: return ntt::fwd_rescale<15>(a, r, s);
        case 16: return ntt::fwd_rescale<16>(a, r, s);
        default: return -2;
    }
}

namespace ntt {
template <int LOGN>
int fwd_dense(const NttArgs* a, pc_stream_t s) {
    if (!a || !a->base || !a->fw || !a->fws || !a->pr || a->xnum < 1 || a->nrows < 0 || a->epi || a->soff) return -1;
    NttArgs A = *a;
    A.roff = nullptr;
    A.rprime = nullptr;
    A.lazy = 0;
    if (A.nrows == 0) return 0;
    if (one_pass(LOGN, A.nrows)) ntt1_fwd(A, 0, A.nrows, s);
    else fwd_pair<LOGN, false>(A, 0, A.nrows, (hipStream_t)s);
    return launch_rc();
}
}  // namespace ntt

bool ntt_one_pass(int logn, int rows) { return ntt::one_pass(logn, rows); }
int ntt_one_pass_min(int rows) {
    const int prev = ntt::ntt1_min();
    ntt::g_ntt1_min.store(rows < 0 ? 0 : rows, std::memory_order_relaxed);
    return prev;
}

int ntt_fwd_dense(int logn, const NttArgs* a, pc_stream_t s) {
    switch (logn) {
        case 12: return ntt::fwd_dense<12>(a, s);
        case 13: return ntt::fwd_dense<13>(a, s);
        case 14: return ntt::fwd_dense<14>(a, s);
        case 15: return ntt::fwd_dense<15>(a, s);
        case 16: return ntt::fwd_dense<16>(a, s);
        default: return -2;
    }
}

int ntt_fwd_rows_only(int logn, const NttArgs* a, pc_stream_t s) {
    switch (logn) {
        case 12: return ntt::fwd_rows_only<12>(a, s);
        case 13: return ntt::fwd_rows_only<13>(a, s);
        case 14: return ntt::fwd_rows_only<14>(a, s);
        case 15: return ntt::fwd_rows_only<15>(a, s);
        case 16: return ntt::fwd_rows_only<16>(a, s);
        default: return -2;
    }
}

#define PCH_NTT_INST(L)                                                             \
    int ntt_fwd_##L(const NttArgs* a, pc_stream_t s) { return ntt::fwd<L>(a, s); } \
    int ntt_inv_##L(const NttArgs* a, pc_stream_t s) { return ntt::inv<L>(a, s); }
PCH_NTT_INST(12)
PCH_NTT_INST(13)
PCH_NTT_INST(14)
PCH_NTT_INST(15)
PCH_NTT_INST(16)

}  // namespace pch
