// Base conversions on the matrix cores, fused into the forward NTT's column pass (mf.h): the words of bconv.hip's jobs
// (prescaled sources) taken through mf_fwd_cols' two steps before they are written, so that a conversion's rows never
// reach memory between the two. mf_ntt_fwd_rows completes the transform.
//
// conv_t = sum_i y_i M[i][t] mod q_t is the contraction of mf.h with the sources as its depth: a word's four bytes times
// (M[i][t] 2^(8a) mod q_t), four targets of four digits as the 16 rows of one MFMA, 16 coefficients as its columns; 16
// sources fill the depth of v_mfma_i32_16x16x64_i8, 8 that of the 16x16x32 form. An output word costs 5 VALU
// instructions where the sums of products took 40 at 16 sources.
//
// A workgroup takes a job's block of 16 columns (R / 16 tiles of 16 rows by 16 columns, two to a wave) and runs of four
// of its targets. Lane (j, q) loads sources NS / 4 q .. of column j's 16 rows tau + (R / 16) k, k = 0 .. 15; the MFMA of
// row k leaves target q's word there. Four lane quarters by four rows transposed in registers (permlane swaps) are the
// first step's vectors: words k = q + 4 v of one target, and the targets are then taken one after the other as
// mf_fwd_cols takes a row. The prime's two matrices (8 KB) and twiddles go through LDS, loaded once per workgroup and
// target, a target ahead.
//
// Bound: latency. 26 ModDowns of C3 (6 sources, 1560 target rows) take 196 us where their 0.58 GB of traffic takes about
// 104: 48% VALU busy (30 instructions per word, 10 of them beside the arithmetic), 19% matrix core, no LDS bank conflicts,
// two workgroups per CU whose waves wait on four chained reads at their start and on a barrier per target. The butterflies'
// form took 265 us (md_conv_cols_k); C3's ModUp 33 -> 21 us, C5's ModUp of four ciphertexts 100 -> 77 us, the exact
// conversion of 8 x 33 rows (bconv_k, then the column pass) 150 -> 74 us. Sources held in registers over all of a
// workgroup's targets (184-254 registers, one workgroup per CU) took 235-340 us for the first.
#include <string.h>

#include "fused.h"
#include "mf.h"
#include "ntt_core.h"

namespace pch {
namespace ntt {

template <int LOGN>
struct Mc {
    using G = Geo<LOGN>;
    static constexpr int R = G::R, C = G::C, T1 = R / 16;
    static constexpr int NT = 2;          // tiles per wave
    static constexpr int W = T1 / NT;     // waves per workgroup
    static constexpr int TH = 64 * W;
    static constexpr int PF = 512 / TH;   // 16-byte words of the two matrices per thread
};
// The exchange of a 16-column group, as MfCol (mfntt.hip) with NT tiles per wave: row r sits at (r, its low two bits xor
// bits 2..3 and 4..5) 16 + column
template <int LOGN>
struct McCol {
    using M = Mc<LOGN>;
    uint32_t s[4], c[4];
    __device__ __forceinline__ McCol(int j, int q, int w) {
        const uint32_t tau = (uint32_t)(M::NT * w);
        const uint32_t ls = M::T1 == 16 ? tau ^ (tau >> 2) ^ q
                            : M::T1 == 8 ? tau ^ (tau >> 2) ^ (2 * (q & 1)) ^ (q >> 1)
                                         : tau ^ q;
        const uint32_t base = (tau & ~3u) + M::T1 * q;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            s[k] = (base + ((k ^ ls) & 3)) * 16 + j;
            c[k] = (16 * tau + 4 * q + ((k ^ q ^ tau) & 3)) * 16 + j;
        }
    }
    // strided: row tau + t + T1 (4 m + q); chunk: row 16 (tau + t) + 4 q + v
    __device__ __forceinline__ uint32_t strided(int t, int m) const {
        return s[(M::T1 == 16 ? t : M::T1 == 8 ? t ^ (2 * (m & 1)) : t ^ m) & 3] + 4 * M::T1 * m * 16;
    }
    __device__ __forceinline__ uint32_t chunk(int t, int v) const { return c[(v ^ t) & 3] + 16 * t * 16; }
};

typedef uint32_t v2u __attribute__((ext_vector_type(2)));
// register r of lane quarter q <- register q of lane quarter r
__device__ __forceinline__ void quarter_transpose(uint32_t& a0, uint32_t& a1, uint32_t& a2, uint32_t& a3) {
    const v2u x = __builtin_amdgcn_permlane32_swap(a0, a2, false, false);
    const v2u y = __builtin_amdgcn_permlane32_swap(a1, a3, false, false);
    const v2u u = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
    const v2u v = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
    a0 = u.x, a1 = u.y, a2 = v.x, a3 = v.y;
}
// mf_reduce with a prime of the lane's own (np = 2^32 - p); also at the 20 sources' depth of 80 (mf.h: r < 1.21 p + 2^29.71)
__device__ __forceinline__ uint32_t mf_reduce_lane(const v4i& s, uint32_t np, uint32_t mu) {
    const uint32_t lo = ((uint32_t)s.y << 8) + (uint32_t)s.x, hi = ((uint32_t)s.w << 8) + (uint32_t)s.z;
    return __umulhi(hi, mu) * np + lshl_add<16>(hi, lo);  // two instructions: v_mad_u64_u32's pairs spill here
}

// a record of eight words, uniform over the wave, in one scalar load
typedef uint32_t v8u __attribute__((ext_vector_type(8)));
template <class T>
__device__ __forceinline__ T sload_rec(const T* p) {
    static_assert(sizeof(T) == 32, "eight words");
    return __builtin_bit_cast(T, sload((const v8u*)p));
}
// tpw: targets per workgroup, 1, 2 or whole runs of four
template <int LOGN, int NS>
__global__ void __launch_bounds__(Mc<LOGN>::TH, LOGN < 14 ? 3 : 4) mf_conv_cols(MfConvArgs A, MfTab T, int tpw) {
    using M = Mc<LOGN>;
    constexpr int NT = M::NT, T1 = M::T1, R = M::R, C = M::C, W = M::W, LW = NS / 4;
    __shared__ uint32_t ex[2][R * 16];
    __shared__ uint4 sm[2][2][256], stw[2][R / 4], sci[2][16], scy[2][8];  // sm: first, second matrices
    const Blk B = blk_xy();
    const int ng = gridDim.x / (C / 16), grp = B.x % ng, cb = B.x / ng;
    // the job's record, source rows and targets at addresses known from the arguments: their reads do not wait for one
    // another
    const uint32_t* jr = A.jobs + (size_t)__builtin_amdgcn_readfirstlane(B.y) * A.stride;
    const MfConvJob J = sload_rec((const MfConvJob*)jr);
    const uint32_t* srow = jr + 8;
    const MfConvTgt* tg = (const MfConvTgt*)(srow + MfConvArgs::src_words(NS));
    const int t0 = tpw * grp, n = min((int)J.nt, t0 + tpw);
    if (t0 >= n) return;  // uniform over the workgroup, before its first barrier
    const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = (uint32_t)(cb * 16 + j);
    uint32_t vs[LW];
#pragma unroll
    for (int v = 0; v < LW; ++v) {
        const int i = v == 4 ? 16 + q : NS == 8 ? 2 * q + v : 4 * q + v;
        vs[v] = (srow[i] << (LOGN + 2)) + (uint32_t)(NT * w * C + col) * 4;
    }
    const Buf bs(A.src + ((size_t)J.src_off << LOGN), J.src_rows << (LOGN + 2));
    const Buf bd(A.dst + ((size_t)J.dst_off << LOGN), J.dst_rows << (LOGN + 2));
    auto ldsrc = [&](int t, int k, uint32_t(&y)[LW]) {
#pragma unroll
        for (int v = 0; v < LW; ++v) y[v] = bs.ld(vs[v], (uint32_t)((t + T1 * k) * C) * 4);
    };
    auto rec = [&](int i) { return sload_rec(tg + min(i, n - 1)); };
    // The matrices, twiddles and initial values: target xi's first matrix, yi's second, each 16-byte word by one thread
    constexpr int PF = M::PF;
    const bool wx = w < W / 2;  // eight waves: the first four take the first matrix
    const uint32_t mk = W == 8 ? threadIdx.x & 255 : threadIdx.x;
    uint4 pm[PF], pt;
    auto fetch = [&](uint32_t xi, uint32_t yi) {
        const uint32_t* mx = T.mat + ((size_t)xi * MF_MATS + MF_X1) * 1024;
        const uint32_t* my = T.mat + ((size_t)yi * MF_MATS + MF_Y1) * 1024;
#pragma unroll
        for (int f = 0; f < PF; ++f) {
            const bool x = W == 8 ? wx : f < PF / 2;
            pm[f] = ((const uint4*)(x ? mx : my))[mk + (PF > 1 ? (int)(f & (PF / 2 - 1)) * M::TH : 0)];
        }
        if (w == 0) {
            if (R == 256 || lane < R / 4) pt = ((const uint4*)(T.tw + (size_t)yi * mf_tw_words(LOGN)))[lane];
        } else if (w == 1 && lane < 24) {
            const uint32_t* ix = T.init + ((size_t)xi * MF_MATS + MF_X1) * 64;
            const uint32_t* iy = T.init + ((size_t)yi * MF_MATS + MF_Y1) * 64;
            pt = lane < 16 ? ((const uint4*)ix)[lane] : ((const uint4*)iy)[lane - 16];
        }
    };
    auto stage = [&](int i) {  // target i's first matrix, target i - 1's second
#pragma unroll
        for (int f = 0; f < PF; ++f) {
            const bool x = W == 8 ? wx : f < PF / 2;
            sm[x ? 0 : 1][(x ? i : i - 1) & 1][mk + (PF > 1 ? (int)(f & (PF / 2 - 1)) * M::TH : 0)] = pm[f];
        }
        if (w == 0) {
            if (R == 256 || lane < R / 4) stw[(i - 1) & 1][lane] = pt;
        } else if (w == 1 && lane < 24) {
            if (lane < 16) sci[i & 1][lane] = pt;
            else scy[(i - 1) & 1][lane - 16] = pt;
        }
    };
    MfConvTgt cur = rec(t0), nxt = rec(t0 + 1);
    fetch(cur.id, cur.id);
    const McCol<LOGN> ck(j, q, w);
    const uint32_t vo = (uint32_t)((16 * NT * w + 4 * q) * C + col) * 4;
    const uint32_t* dig = A.dig + J.dig + (size_t)(t0 / 4) * MfConvArgs::group_words(NS);
    for (int g = t0 & ~3; g < n; g += 4, dig += MfConvArgs::group_words(NS)) {
        // the run's words of its four targets
        uint32_t x[NT][4][4];  // [target][v] after the transpose
        {
            const MfConvTgt* lt = tg + min(g + q, (int)J.nt - 1);
            const uint32_t np = 0u - lt->p, mu = lt->mu;
            v4i a0 = {}, a1 = {};
            long h0 = 0;
            if constexpr (NS == 8) h0 = ((const long*)dig)[lane];
            else a0 = ((const v4i*)dig)[lane];
            if constexpr (NS == 20) a1.x = (int)dig[256 + lane];
            const v4i ci = ((const v4i*)(dig + NS * 16))[q];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    uint32_t r[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        uint32_t s[LW];
                        ldsrc(t, u + 4 * v, s);
                        v4i d = ci;
                        if constexpr (NS >= 16) {
                            const v4i b = {(int)(s[0] ^ MF_FLIP), (int)(s[1] ^ MF_FLIP), (int)(s[2] ^ MF_FLIP),
                                           (int)(s[3] ^ MF_FLIP)};
                            d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b, d, 0, 0, 0);
                        }
                        if constexpr (NS == 20) {
                            // not the 16x16x32 form: the compiler issues it right behind the 16x16x64 whose result it
                            // accumulates onto, and half its words then miss that result (alone, 128 of 256 words
                            // wrong back to back, none with wait states between or with the two sums added)
                            const v4i b = {(int)(s[4] ^ MF_FLIP), 0, 0, 0};
                            d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b, d, 0, 0, 0);
                        }
                        if constexpr (NS == 8) {
                            const uint64_t b = ((uint64_t)(s[1] ^ MF_FLIP) << 32) | (s[0] ^ MF_FLIP);
                            d = __builtin_amdgcn_mfma_i32_16x16x32_i8(h0, (long)b, d, 0, 0, 0);
                        }
                        r[u] = mf_reduce_lane(d, np, mu);
                    }
                    quarter_transpose(r[0], r[1], r[2], r[3]);
#pragma unroll
                    for (int u = 0; u < 4; ++u) x[t][u][v] = r[u];
                }
        }
        if (g <= t0) {  // the first run: its matrices came in with the sources
            stage(t0);
            fetch(nxt.id, cur.id);
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = g + u;
            if (i < t0) continue;
            if (i >= n) break;
            const MfPrime P(cur.p, cur.mu, cur.pinv);
            const MfConvTgt nn = rec(i + 2);
            {
                MfMat X;
                MfInit<true> cx;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    X.a[k] = ((const v4i*)sm[0][u & 1])[64 * k + lane];
                    cx.c[k] = ((const v4i*)sci[u & 1])[4 * k + q];
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    mf_apply(x[t][u], X, cx, P);
#pragma unroll
                    for (int m = 0; m < 4; ++m) ex[u & 1][ck.strided(t, m)] = x[t][u][m];
                }
            }
            stage(i + 1);
            __syncthreads();
            if (i + 1 < n) fetch(nn.id, nxt.id);
            MfMat Y;
            MfInit<false> cy;
            cy.c[0] = ((const v4i*)scy[u & 1])[q];
            cy.c[1] = ((const v4i*)scy[u & 1])[4 + q];
#pragma unroll
            for (int k = 0; k < 4; ++k) Y.a[k] = ((const v4i*)sm[1][u & 1])[64 * k + lane];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                uint32_t z[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) z[v] = ex[u & 1][ck.chunk(t, v)];
                mf_twist(z, stw[u & 1][4 * (NT * w + t) + q], P);
                mf_apply(z, Y, cy, P);
#pragma unroll
                for (int m = 0; m < 4; ++m) bd.st(z[m], vo, ((cur.row << LOGN) + (uint32_t)((16 * t + m) * C)) * 4);
            }
            cur = nxt, nxt = nn;
        }
    }
}

// The exact jobs' quotients, once per coefficient (bconv_k and conv_cols_k form them per group of targets). Two
// coefficients per thread: a product's four rows of N = 2^16 are then 512 workgroups.
__global__ void __launch_bounds__(256) conv_u_k(BconvArgs A, uint32_t* u, int logn) {
    const BconvJob* jp = A.jobs + blockIdx.y;
    const int ns = (int)sload(&jp->nsrc), nt = (int)sload(&jp->ntgt);
    const uint32_t* pool = (const uint32_t*)A.pool + sload(&jp->pool_off);
    size_t w = (size_t)sload(&jp->pool_off) + 3 * ns + 2 * nt + (size_t)ns * nt;
    if (w & 1) ++w;
    const double* rb = (const double*)((const uint32_t*)A.pool + w);
    const size_t o = ((size_t)blockIdx.x * 256 + threadIdx.x) * 2;
    const uint32_t* src = (const uint32_t*)A.src + ((size_t)sload(&jp->src_off) << logn) + o;
    double v0 = 0.0, v1 = 0.0;
    for (int i0 = 0; i0 < ns; i0 += MFC_MAX_NS) {
        uint2 y[MFC_MAX_NS];
#pragma unroll
        for (int i = 0; i < MFC_MAX_NS; ++i)
            if (i0 + i < ns) y[i] = *(const uint2*)(src + ((size_t)sload(pool + i0 + i) << logn));
#pragma unroll
        for (int i = 0; i < MFC_MAX_NS; ++i)
            if (i0 + i < ns) {
                const double r = sload(rb + i0 + i);
                v0 = __fma_rn((double)y[i].x, r, v0);
                v1 = __fma_rn((double)y[i].y, r, v1);
            }
    }
    *(uint2*)(u + ((size_t)blockIdx.y << logn) + o) =
        make_uint2((uint32_t)(uint64_t)floor(v0 + 0.5), (uint32_t)(uint64_t)floor(v1 + 0.5));
}

template <int LOGN, int NS>
int mfc_launch(const MfConvArgs& a, const MfTab& t, int tpw, hipStream_t st) {
    using M = Mc<LOGN>;
    const int ng = (a.max_tgt + tpw - 1) / tpw;
    hipLaunchKernelGGL((mf_conv_cols<LOGN, NS>), dim3(M::C / 16 * ng, a.njobs), dim3(M::TH), 0, st, a, t, tpw);
    return launch_rc();
}
template <int LOGN>
int mfc(const MfConvArgs* a, const MfTab* t, int tpw, pc_stream_t s) {
    if (!a || !t || !a->src || !a->dst || !a->jobs || !a->dig || a->njobs < 0) return -1;
    if (!t->tw || !t->mat || !t->init || t->can < 1) return -1;
    if (a->njobs > 65535 || a->max_tgt < 1 || tpw < 1 || (tpw > 2 && tpw % 4)) return -1;
    if (a->njobs == 0) return 0;
    switch (a->ns) {
        case 8: return mfc_launch<LOGN, 8>(*a, *t, tpw, (hipStream_t)s);
        case 16: return mfc_launch<LOGN, 16>(*a, *t, tpw, (hipStream_t)s);
        case 20: return mfc_launch<LOGN, 20>(*a, *t, tpw, (hipStream_t)s);
        default: return -2;
    }
}

}  // namespace ntt

int mf_conv_cols(int logn, const MfConvArgs* a, const MfTab* t, int tpw, pc_stream_t s) {
    switch (logn) {
        case 12: return ntt::mfc<12>(a, t, tpw, s);
        case 13: return ntt::mfc<13>(a, t, tpw, s);
        case 14: return ntt::mfc<14>(a, t, tpw, s);
        case 15: return ntt::mfc<15>(a, t, tpw, s);
        case 16: return ntt::mfc<16>(a, t, tpw, s);
        default: return -2;
    }
}

int conv_u(int logn, const BconvArgs* a, uint32_t* u, pc_stream_t s) {
    if (!a || !u || !a->src || !a->jobs || !a->pool || a->njobs < 0 || a->njobs > 65535) return -1;
    if (logn < 12 || logn > 16) return -2;
    if (a->njobs == 0) return 0;
    hipLaunchKernelGGL(ntt::conv_u_k, dim3((1u << logn) / 512, a->njobs), dim3(256), 0, (hipStream_t)s, *a, u, logn);
    return launch_rc();
}

// the digits of one group of at most four targets: w[i][t] = M[i][t] mod p[t], nt targets, n sources of ns
void mf_conv_digits(const uint64_t* w, int n, int nt, const uint64_t* p, int ns, uint32_t* out) {
    memset(out, 0, MfConvArgs::group_words(ns) * 4);
    int8_t* b = (int8_t*)out;
    const uint64_t B = ns > 16 ? 1u << 21 : 1u << 20, ones = 0x01010101ull;
    for (int t = 0; t < nt; ++t) {
        uint64_t sum = 0;
        for (int i = 0; i < n; ++i) {
            // source i: byte a of word v of lane quarter q
            const bool hi = i >= 16;
            const int ii = hi ? i - 16 : i, per = hi ? 1 : ns == 8 ? 2 : 4;
            int8_t* blk = b + (hi ? 1024 : 0);
            for (int a = 0; a < 4; ++a) {
                const uint64_t m = w[i * nt + t] * ((1ull << (8 * a)) % p[t]) % p[t];
                sum = (sum + m) % p[t];
                int8_t d[4];
                mf_digits(m, p[t], d);
                for (int k = 0; k < 4; ++k) blk[((16 * (ii / per) + 4 * t + k) * per + ii % per) * 4 + a] = d[k];
            }
        }
        // sum_i c_i 2^(8i) == 128 sum W (mod p) with c_i = B + d_i, B >= the largest |sum| of a digit's products (2^20 at depth
        // 64, 1.25 2^20 at 80)
        const uint64_t need = (sum * 128 + p[t] - B * ones % p[t]) % p[t];
        for (int k = 0; k < 4; ++k) out[ns * 16 + 4 * t + k] = (uint32_t)(B + ((need >> (8 * k)) & 255));
    }
}

}  // namespace pch
