// The NTT passes on the matrix cores (mf.h): the transforms of ntt.hip, the same words, each radix-16 step one int8 MFMA
// contraction instead of four butterfly stages.
//
// A row of N = R x C words is transformed as in ntt.hip: a column pass over the R-point columns, a row pass over the
// C-word blocks, two steps each (radix 16, then R / 16 or C / 16). The unit of work of a wave is a tile of 16 vectors of
// 16 words: lane (j, q), j = lane mod 16 and q = lane / 16, holds four words of vector j.
//  Column pass: a tile is 16 columns by 16 rows; step 1 takes rows tau + (R / 16) k, k = q + 4 v (outputs 4 m + q), the
//   workgroup's tiles are exchanged through LDS, step 2 takes 16 consecutive rows 16 b + 4 q + v (outputs 4 q + m).
//  Row pass: a tile is 256 consecutive words; step 1 takes its 16-word vectors at stride C / 16 (k = q + 4 v: each load
//   instruction covers 256 consecutive bytes), the tile is transposed through LDS within the wave, step 2 takes 16
//   consecutive words (4 q + v, outputs 4 q + m: 16-byte accesses that cover the tile).
// The inverse runs the same steps backwards.
//
// Bound: the words' two moves through memory. 2560 rows of N = 2^16 at 31-bit primes: 556 us forward, 546 us inverse (4.8
// TB/s over the two passes) against 580 and 605 us for the butterflies of ntt.hip, which were 81-85% VALU busy; 102
// rows inverse 25.4 against 29.1 us (same box). Four tiles per wave give a wave's loads something to hide behind
// without keeping the matrices (4 KB each, from L1 / L2) for more words: two or four rounds of tiles per workgroup took
// 566-586 us. Twiddle tables of N words per prime, one or two per data word, took 690 us: the vector memory path, not the
// VALU, is what a pass must be spared.
#include <string.h>

#include <vector>

#include "fused.h"
#include "mf.h"
#include "ntt_core.h"

namespace pch {
namespace ntt {

constexpr int MW = 4;    // waves per workgroup
constexpr int MT = 4;    // tiles per wave

template <int LOGN>
struct Mg {
    using G = Geo<LOGN>;
    static constexpr int N = G::N, R = G::R, C = G::C;
    static constexpr int T1 = R / 16;             // column tiles of a 16-column group
    static constexpr int CG = MW * MT / T1;       // 16-column groups of a workgroup
    static constexpr int COLS = 16 * CG;          
    static constexpr int S = C / 16;              // stride of a row pass's first step
    static constexpr int TB = 256 / C;            // blocks of a row tile
    static constexpr int LDS = MW * MT * 256;     // words of a workgroup
    static constexpr uint32_t TW1 = 0, TW2 = R, TWB = 17 * R, XI = 33 * R, TWN = mf_tw_words(LOGN);
    static_assert(CG >= 1 && C % COLS == 0 && N % LDS == 0, "whole workgroups");
};
// A column workgroup's exchange. Row r of a 16-column group sits at (r with its low two bits mixed with bits 2..3 and 4..5)
// 16 + column, so that the four rows that a wave touches at once (4 apart on one side, R / 16 apart on the other) sit
// in four distinct 16-bank blocks on both sides. The low bits are a compile-time part xor a lane's part: a lane needs
// four addresses per side, and the rest of a row is an immediate offset.
template <int LOGN>
struct MfCol {
    using M = Mg<LOGN>;
    uint32_t s[4], c[4];
    // tile t of wave w is column group (4 w + t) / T1, number (4 w + t) mod T1 = 4 (w mod (T1 / 4)) + t
    __device__ __forceinline__ MfCol(int j, int q, int w) {
        constexpr int W4 = M::T1 / 4;
        const uint32_t cg = (uint32_t)(w / W4) * M::R, w4 = 4 * (uint32_t)(w % W4);
        const uint32_t ls = M::T1 == 16 ? w ^ q : M::T1 == 8 ? ((w & 1) ^ (q >> 1)) | ((q & 1) << 1) : q;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            s[k] = (cg + w4 + M::T1 * q + ((k ^ ls) & 3)) * 16 + j;
            c[k] = (cg + 16 * w4 + 4 * q + ((k ^ q) & 3)) * 16 + j;
        }
    }
    // strided: row tau + T1 (4 m + q) of tile t
    __device__ __forceinline__ uint32_t strided(int t, int m) const {
        return s[(M::T1 == 16 ? t : M::T1 == 8 ? t ^ (2 * (m & 1)) : t ^ m) & 3] + 4 * M::T1 * m * 16;
    }
    // chunk: row 16 b + 4 q + v of tile t
    __device__ __forceinline__ uint32_t chunk(int t, int v) const { return c[(v ^ t) & 3] + 16 * t * 16; }
    // the tile's number tau = b
    static __device__ __forceinline__ int tile(int w, int t) { return 4 * (w % (M::T1 / 4)) + t; }
    static __device__ __forceinline__ int group(int w) { return w / (M::T1 / 4); }
};
// A row tile's word at position pos: the 4-word quarters of each 16-word chunk permuted by the chunk's number, so that
// both the 16-byte accesses (a chunk per lane) and the word accesses of 64 consecutive positions are conflict-free
__device__ __forceinline__ uint32_t mf_pos(uint32_t pos) {
    const uint32_t g = pos >> 4;
    return (pos & ~12u) | ((((pos >> 2) ^ (g >> 2)) & 3u) << 2);
}

struct MfLane {
    int lane, j, q, w;
    __device__ __forceinline__ MfLane()
        : lane(threadIdx.x & 63), j(lane & 15), q(lane >> 4), w(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {}
};
__device__ __forceinline__ uint4 ld4(const uint32_t* p) { return *(const uint4*)p; }

// ------------------------------------------------------------------------------------------------ column passes
// Workgroup (x, row): COLS columns from column x COLS.
// GEN: the rows are rescale corrections generated by RsGen from R
template <int LOGN, bool GEN = false>
__global__ void __launch_bounds__(64 * MW, 4) mf_fwd_cols(NttArgs A, MfTab T, int row0, RescaleArgs R = {}) {
    using M = Mg<LOGN>;
    using K = MfCol<LOGN>;
    __shared__ uint32_t lds[M::LDS], ltw[M::R];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const uint32_t* row = (const uint32_t*)A.base + (row_off(A, i) << LOGN);
    const Buf bs(GEN || !A.soff ? row : (const uint32_t*)A.src + ((size_t)A.soff[i] << LOGN), (uint32_t)M::N * 4);
    const Buf bo(row, (uint32_t)M::N * 4);
    const uint32_t c0 = (uint32_t)(B.x * M::COLS + K::group(L.w) * 16 + L.j);
    const uint32_t vi = (K::tile(L.w, 0) + M::T1 * L.q) * M::C + c0, vo = (16 * K::tile(L.w, 0) + 4 * L.q) * M::C + c0;
    uint32_t x[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t so = (uint32_t)((t + M::T1 * 4 * v) * M::C);
            if constexpr (GEN) x[t][v] = RsGen(R, row, pid, LOGN)(vi + so);
            else x[t][v] = bs.ld(vi * 4, so * 4);
        }
    MfMat X, Y;
    MfInit<true> cx;
    MfInit<false> cy;
    X.load(T, pid, MF_X1, L.lane);
    cx.template load<16>(T, pid, MF_X1, L.lane);
    Y.load(T, pid, MF_Y1, L.lane);
    cy.template load<M::T1>(T, pid, MF_Y1, L.lane);
    if (threadIdx.x < M::R / 4)
        ((uint4*)ltw)[threadIdx.x] = ld4(T.tw + (size_t)pid * M::TWN + M::TW1 + 4 * threadIdx.x);
    const K k(L.j, L.q, L.w);
    const uint32_t* lt = ltw + 16 * K::tile(L.w, 0) + 4 * L.q;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        mf_apply(x[t], X, cx, P);
#pragma unroll
        for (int m = 0; m < 4; ++m) lds[k.strided(t, m)] = x[t][m];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        uint32_t y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = lds[k.chunk(t, v)];
        mf_twist(y, ld4(lt + 16 * t), P);
        mf_apply(y, Y, cy, P);
#pragma unroll
        for (int m = 0; m < 4; ++m) bo.st(y[m], vo * 4, (uint32_t)((16 * t + m) * M::C) * 4);
    }
}

template <int LOGN>
__global__ void __launch_bounds__(64 * MW, 4) mf_inv_cols(NttArgs A, MfTab T, int row0) {
    using M = Mg<LOGN>;
    using K = MfCol<LOGN>;
    __shared__ uint32_t lds[M::LDS], ltw[M::R];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const Buf ba((const uint32_t*)A.base + (row_off(A, i) << LOGN), (uint32_t)M::N * 4);
    const uint32_t c0 = (uint32_t)(B.x * M::COLS + K::group(L.w) * 16 + L.j);
    const uint32_t vo = (K::tile(L.w, 0) + M::T1 * L.q) * M::C + c0, vi = (16 * K::tile(L.w, 0) + 4 * L.q) * M::C + c0;
    uint32_t x[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) x[t][v] = ba.ld(vi * 4, (uint32_t)((16 * t + v) * M::C) * 4);
    MfMat X, Y;
    MfInit<true> cx;
    MfInit<false> cy;
    Y.load(T, pid, MF_INV + MF_Y1, L.lane);
    cy.template load<M::T1>(T, pid, MF_INV + MF_Y1, L.lane);
    X.load(T, pid, MF_INV + MF_X1, L.lane);
    cx.template load<16>(T, pid, MF_INV + MF_X1, L.lane);
    if (threadIdx.x < M::R / 4)
        ((uint4*)ltw)[threadIdx.x] = ld4(T.itw + (size_t)pid * M::TWN + M::TW1 + 4 * threadIdx.x);
    // the scale: es[i] per row (NttArgs ABI 17) or N^-1 of the prime
    const uint32_t s = A.es ? sload((const uint32_t*)A.es + i) : sload((const uint32_t*)A.ninv + pid);
    const uint32_t ss = A.es ? sload((const uint32_t*)A.ess + i) : sload((const uint32_t*)A.ninvs + pid);
    const K k(L.j, L.q, L.w);
    const uint32_t* lt = ltw + 16 * K::tile(L.w, 0) + 4 * L.q;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        mf_apply(x[t], Y, cy, P);
        mf_twist(x[t], ld4(lt + 16 * t), P);
#pragma unroll
        for (int m = 0; m < 4; ++m) lds[k.chunk(t, m)] = x[t][m];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        uint32_t y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = lds[k.strided(t, v)];
        mf_apply(y, X, cx, P);
#pragma unroll
        for (int m = 0; m < 4; ++m)
            ba.st(shoup(y[m], s, ss, P.p), vo * 4, (uint32_t)((t + M::T1 * 4 * m) * M::C) * 4);
    }
}

// ------------------------------------------------------------------------------------------------ row passes
// Workgroup (x, row): its waves take MT tiles each, consecutive in the row. The 32 twiddles of each of the wave's blocks
// go through LDS, which serves a tile's lanes their quarter's four at once.
template <int LOGN>
struct MfRowTw {
    using M = Mg<LOGN>;
    static constexpr int BLKS = MT * M::TB;      // the wave's blocks
    static constexpr int WORDS = 2 * 16 * BLKS;       // TW2 then TWB of each
    // the wave's blocks from blk0 on, staged by the wave
    static __device__ __forceinline__ void stage(uint32_t* l, const uint32_t* tw, uint32_t blk0, int lane) {
        for (int k = lane; k < BLKS * 4; k += 64) {
            ((uint4*)l)[k] = ((const uint4*)(tw + M::TW2 + blk0 * 16))[k];
            ((uint4*)l)[BLKS * 4 + k] = ((const uint4*)(tw + M::TWB + blk0 * 16))[k];
        }
    }
};
template <int LOGN, int EPI, int CAN>
__global__ void __launch_bounds__(64 * MW, 4) mf_fwd_rows(NttArgs A, MfTab T, int row0) {
    using M = Mg<LOGN>;
    using W = MfRowTw<LOGN>;
    __shared__ uint32_t lds[M::LDS], ltw[MW][W::WORDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const size_t row = row_off(A, i) << LOGN;
    const uint32_t o0 = (uint32_t)(B.x * MW + L.w) * MT * 256;  // the wave's first word in the row
    const int bl = L.j / M::S, jj = L.j % M::S;  // vector j of a tile: block bl, offset jj
    typedef const __attribute__((address_space(1))) uint32_t* gp;
    const gp a = (gp)((const uint32_t*)A.base + row + o0 + bl * M::C + L.q * M::S + jj);
    uint32_t x[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const gp p = a + t * 256 + 4 * v * M::S;
            x[t][v] = EPI ? __builtin_nontemporal_load(p) : *p;
        }
    const uint32_t* tw = T.tw + (size_t)pid * M::TWN;
    uint32_t* lt = ltw[L.w];
    W::stage(lt, tw, o0 / M::C, L.lane);
    MfMat X, Y;
    MfInit<false> cx, cy;
    X.load(T, pid, MF_X16, L.lane);
    cx.template load<16>(T, pid, MF_X16, L.lane);
    Y.load(T, pid, MF_Y2, L.lane);
    cy.template load<M::S>(T, pid, MF_Y2, L.lane);
    const uint32_t pos = 16 * L.j + 4 * L.q;
    const uint4 xi = ld4(tw + M::XI + pos % M::C);
    uint32_t s = 0, ss = 0;
    if (EPI) s = sload((const uint32_t*)A.es + pid), ss = sload((const uint32_t*)A.ess + pid);
    uint32_t* l = lds + L.w * MT * 256;
    wave_sync();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        mf_twist(x[t], ld4(lt + (t * M::TB + bl) * 16 + 4 * L.q), P);
        mf_apply(x[t], X, cx, P);
#pragma unroll
        for (int m = 0; m < 4; ++m) l[t * 256 + mf_pos(bl * M::C + (4 * m + L.q) * M::S + jj)] = x[t][m];
    }
    wave_sync();
    // the epilogue's operand, every word of the wave in flight before the second step; read once: past the caches
    typedef const __attribute__((address_space(1))) gu4* gq;
    const uint32_t* exb = (const uint32_t*)A.ex + row + o0 + pos;
    gu4 ex[MT];
    if (EPI) {
#pragma unroll
        for (int t = 0; t < MT; ++t) ex[t] = __builtin_nontemporal_load((gq)(exb + t * 256));
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const uint4 y4 = ld4(l + t * 256 + mf_pos(pos));
        uint32_t y[4] = {y4.x, y4.y, y4.z, y4.w};
        mf_twist(y, xi, P);
        mf_twist(y, ld4(lt + W::WORDS / 2 + (t * M::TB + pos / M::C) * 16 + 4 * L.q), P);
        mf_apply(y, Y, cy, P);
        const size_t r0 = row + o0 + t * 256 + pos;
        uint4 z = make_uint4(mf_canon<CAN>(y[0], P), mf_canon<CAN>(y[1], P), mf_canon<CAN>(y[2], P),
                             mf_canon<CAN>(y[3], P));
        if (EPI == 0) {
            *(uint4*)((uint32_t*)A.base + r0) = z;
            continue;
        }
        for (int k = 1; k < A.xnum; ++k) {
            const uint4 e = ld4(exb + t * 256 + k * A.xstride);
            ex[t].x = addm(ex[t].x, e.x, P.p), ex[t].y = addm(ex[t].y, e.y, P.p);
            ex[t].z = addm(ex[t].z, e.z, P.p), ex[t].w = addm(ex[t].w, e.w, P.p);
        }
        uint32_t* eo = (uint32_t*)A.eout + r0;
        uint4 d = make_uint4(0, 0, 0, 0);
        if (EPI == 2) d = ld4(A.ed ? (const uint32_t*)A.ed + r0 : eo);
        auto fin = [&](uint32_t v, uint32_t e, uint32_t dd) {
            if (EPI == 3) return addm(shoup(e, s, ss, P.p), v, P.p);
            const uint32_t y1 = shoup(e - v + P.p, s, ss, P.p);
            return EPI == 2 ? addm(dd, y1, P.p) : y1;
        };
        z = make_uint4(fin(z.x, ex[t].x, d.x), fin(z.y, ex[t].y, d.y), fin(z.z, ex[t].z, d.z), fin(z.w, ex[t].w, d.w));
        *(uint4*)eo = z;
    }
}

template <int LOGN>
__global__ void __launch_bounds__(64 * MW, 4) mf_inv_rows(NttArgs A, MfTab T, int row0) {
    using M = Mg<LOGN>;
    using W = MfRowTw<LOGN>;
    __shared__ uint32_t lds[M::LDS], ltw[MW][W::WORDS];
    const Blk B = blk_xy();
    const int i = row0 + B.y;
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const RowSrc src = row_src(A, i, LOGN);
    const uint32_t o0 = (uint32_t)(B.x * MW + L.w) * MT * 256;
    const uint32_t pos = 16 * L.j + 4 * L.q;
    const uint32_t* sp = src.p0 + o0 + pos;
    uint4 x[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) x[t] = ld4(sp + t * 256);
    for (int k = 1; k < src.n; ++k)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint4 e = ld4(sp + k * src.stride + t * 256);
            x[t].x = addm(x[t].x, e.x, P.p), x[t].y = addm(x[t].y, e.y, P.p);
            x[t].z = addm(x[t].z, e.z, P.p), x[t].w = addm(x[t].w, e.w, P.p);
        }
    const uint32_t* tw = T.itw + (size_t)pid * M::TWN;
    uint32_t* lt = ltw[L.w];
    W::stage(lt, tw, o0 / M::C, L.lane);
    MfMat X, Y;
    MfInit<false> cx, cy;
    Y.load(T, pid, MF_INV + MF_Y2, L.lane);
    cy.template load<M::S>(T, pid, MF_INV + MF_Y2, L.lane);
    X.load(T, pid, MF_INV + MF_X16, L.lane);
    cx.template load<16>(T, pid, MF_INV + MF_X16, L.lane);
    const uint4 xi = ld4(tw + M::XI + pos % M::C);
    uint32_t* l = lds + L.w * MT * 256;
    const int bl = L.j / M::S, jj = L.j % M::S;
    uint32_t* o = (uint32_t*)A.base + (row_off(A, i) << LOGN) + o0 + bl * M::C + L.q * M::S + jj;
    wave_sync();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        uint32_t y[4] = {x[t].x, x[t].y, x[t].z, x[t].w};
        mf_apply(y, Y, cy, P);
        mf_twist(y, xi, P);
        mf_twist(y, ld4(lt + W::WORDS / 2 + (t * M::TB + pos / M::C) * 16 + 4 * L.q), P);
        *(uint4*)(l + t * 256 + mf_pos(pos)) = make_uint4(y[0], y[1], y[2], y[3]);
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        uint32_t y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = l[t * 256 + mf_pos(bl * M::C + (4 * v + L.q) * M::S + jj)];
        mf_apply(y, X, cx, P);
        mf_twist(y, ld4(lt + (t * M::TB + bl) * 16 + 4 * L.q), P);
#pragma unroll
        for (int m = 0; m < 4; ++m) o[t * 256 + 4 * m * M::S] = y[m];
    }
}

// ------------------------------------------------------------------------------------------------ one pass
// Rows of at most 2^14 words stay in one workgroup's LDS between the column and the row pass: a launch instead of two, and
// each word read and written once. The tiles and steps are the two passes'. GEN: as mf_fwd_cols (RsGen).
//
// Bound: small launches by their chain of reads and barriers (12 rows of N = 2^12: 5.7 us, the two passes 7.6; of 2^13 7.2
// and 8.0), large ones by the VALU (1600 rows of N = 2^14: 62 us, the two passes 72). One row of N = 2^14 is eight tiles for
// each of its CU's waves: 10.6 us where the two passes spread it over several CUs and take 7.8. Up to 256 rows have a CU each
// and up to 512 half of one, so its time is a stair of steps at those counts (one launch / two passes, forward, us: 128 rows
// 12.4 / 11.4, 144 12.6 / 13.3, 256 13.6 / 16.9, 257 18.8 / 18.2, 320 19.9 / 18.9, 336 19.9 / 20.6, 512 21.0 / 27.0, 513
// 27.3 / 28.2, 2560 96 / 111): it is taken for 129 to 256 rows and above 320 (one14).
inline bool one14(int rows) { return (rows > 128 && rows <= 256) || rows > 320; }
template <int LOGN>
struct Mo {
    using M = Mg<LOGN>;
    static constexpr int T = M::N / 256;            // tiles
    static constexpr int MT = LOGN == 14 ? 8 : 4;   // per wave
    static constexpr int W = T / MT;
    // Word (r, c) of the row sits at r C + (c with its 16-word block xor g(r)): the four rows that a column step's wave
    // touches at once (4 apart, R / 16 apart) and the two or four rows of a row tile then sit in distinct blocks
    static __device__ __forceinline__ uint32_t pos(uint32_t r, uint32_t c) {
        const uint32_t g = M::C == 128 ? ((r >> 2) & 3) ^ ((r >> 4) & (M::T1 == 8 ? 1 : 3)) ^ ((r & 1) << 1)
                                       : ((r >> 2) & 3) ^ ((r >> 4) & 3) ^ (r & 3);
        return r * M::C + (c ^ (g << 4));
    }
};
// Four consecutive words at offset o of a (its row and position in it) through the epilogue
template <int EPI, int CAN>
__device__ __forceinline__ void mf_out(const NttArgs& A, size_t o, const uint32_t (&y)[4], uint32_t s, uint32_t ss,
                                       const MfPrime& P) {
    uint4 z = make_uint4(mf_canon<CAN>(y[0], P), mf_canon<CAN>(y[1], P), mf_canon<CAN>(y[2], P), mf_canon<CAN>(y[3], P));
    if (EPI == 0) {
        *(uint4*)((uint32_t*)A.base + o) = z;
        return;
    }
    const uint32_t* exb = (const uint32_t*)A.ex + o;
    uint4 ex = ld4(exb);
    for (int k = 1; k < A.xnum; ++k) {
        const uint4 e = ld4(exb + k * A.xstride);
        ex.x = addm(ex.x, e.x, P.p), ex.y = addm(ex.y, e.y, P.p);
        ex.z = addm(ex.z, e.z, P.p), ex.w = addm(ex.w, e.w, P.p);
    }
    uint32_t* eo = (uint32_t*)A.eout + o;
    uint4 d = make_uint4(0, 0, 0, 0);
    if (EPI == 2) d = ld4(A.ed ? (const uint32_t*)A.ed + o : eo);
    auto fin = [&](uint32_t v, uint32_t e, uint32_t dd) {
        if (EPI == 3) return addm(shoup(e, s, ss, P.p), v, P.p);
        const uint32_t y1 = shoup(e - v + P.p, s, ss, P.p);
        return EPI == 2 ? addm(dd, y1, P.p) : y1;
    };
    *(uint4*)eo = make_uint4(fin(z.x, ex.x, d.x), fin(z.y, ex.y, d.y), fin(z.z, ex.z, d.z), fin(z.w, ex.w, d.w));
}
template <int LOGN, int EPI, int CAN, bool GEN = false>
__global__ void __launch_bounds__(64 * Mo<LOGN>::W, 4) mf_fwd_one(NttArgs A, MfTab T, RescaleArgs R = {}) {
    using O = Mo<LOGN>;
    using M = Mg<LOGN>;
    constexpr int MT = O::MT;
    __shared__ uint32_t lds[M::N];
    const int i = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const size_t row = row_off(A, i) << LOGN;
    const Buf bs(A.soff ? (const uint32_t*)A.src + ((size_t)A.soff[i] << LOGN) : (const uint32_t*)A.base + row,
                 (uint32_t)M::N * 4);
    const uint32_t* tw = T.tw + (size_t)pid * M::TWN;
    {
        const uint32_t tau = (uint32_t)(L.w * MT % M::T1), col = (uint32_t)(L.w * MT / M::T1 * 16 + L.j);
        uint32_t x[MT][4];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t vo = (tau + M::T1 * L.q) * M::C + col, so = (uint32_t)((t + M::T1 * 4 * v) * M::C);
                if constexpr (GEN) x[t][v] = RsGen(R, (const uint32_t*)A.base + row, pid, LOGN)(vo + so);
                else x[t][v] = bs.ld(vo * 4, so * 4);
            }
        MfMat X, Y;
        MfInit<true> cx;
        MfInit<false> cy;
        X.load(T, pid, MF_X1, L.lane);
        cx.template load<16>(T, pid, MF_X1, L.lane);
        Y.load(T, pid, MF_Y1, L.lane);
        cy.template load<M::T1>(T, pid, MF_Y1, L.lane);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            mf_apply(x[t], X, cx, P);
#pragma unroll
            for (int m = 0; m < 4; ++m) lds[O::pos(tau + t + M::T1 * (4 * m + L.q), col)] = x[t][m];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint32_t r = 16 * (tau + t) + 4 * L.q;
            uint32_t y[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) y[v] = lds[O::pos(r + v, col)];
            mf_twist(y, ld4(tw + M::TW1 + r), P);
            mf_apply(y, Y, cy, P);
            // the wave's own words, read by no other before the barrier
#pragma unroll
            for (int m = 0; m < 4; ++m) lds[O::pos(r + m, col)] = y[m];
        }
    }
    MfMat X, Y;
    MfInit<false> cx, cy;
    X.load(T, pid, MF_X16, L.lane);
    cx.template load<16>(T, pid, MF_X16, L.lane);
    Y.load(T, pid, MF_Y2, L.lane);
    cy.template load<M::S>(T, pid, MF_Y2, L.lane);
    const uint32_t pos = 16 * L.j + 4 * L.q;
    const uint4 xi = ld4(tw + M::XI + pos % M::C);
    uint32_t s = 0, ss = 0;
    if (EPI) s = sload((const uint32_t*)A.es + pid), ss = sload((const uint32_t*)A.ess + pid);
    const int bl = L.j / M::S, jj = L.j % M::S;
    const uint32_t b0 = (uint32_t)(L.w * MT * M::TB);  // the wave's first block
    __syncthreads();
    uint32_t x[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) x[t][v] = lds[O::pos(b0 + t * M::TB + bl, (4 * v + L.q) * M::S + jj)];
    wave_sync();
    uint32_t* l = lds + L.w * MT * 256;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        mf_twist(x[t], ld4(tw + M::TW2 + (b0 + t * M::TB + bl) * 16 + 4 * L.q), P);
        mf_apply(x[t], X, cx, P);
#pragma unroll
        for (int m = 0; m < 4; ++m) l[t * 256 + mf_pos(bl * M::C + (4 * m + L.q) * M::S + jj)] = x[t][m];
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const uint4 y4 = ld4(l + t * 256 + mf_pos(pos));
        uint32_t y[4] = {y4.x, y4.y, y4.z, y4.w};
        mf_twist(y, xi, P);
        mf_twist(y, ld4(tw + M::TWB + (b0 + t * M::TB + pos / M::C) * 16 + 4 * L.q), P);
        mf_apply(y, Y, cy, P);
        mf_out<EPI, CAN>(A, row + (L.w * MT + t) * 256 + pos, y, s, ss, P);
    }
}

template <int LOGN>
__global__ void __launch_bounds__(64 * Mo<LOGN>::W, 4) mf_inv_one(NttArgs A, MfTab T) {
    using O = Mo<LOGN>;
    using M = Mg<LOGN>;
    constexpr int MT = O::MT;
    __shared__ uint32_t lds[M::N];
    const int i = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x));
    const int pid = __builtin_amdgcn_readfirstlane(row_prime(A, i));
    const MfLane L;
    const MfPrime P(A.pr, pid);
    const RowSrc src = row_src(A, i, LOGN);
    const uint32_t* tw = T.itw + (size_t)pid * M::TWN;
    const uint32_t pos = 16 * L.j + 4 * L.q;
    const uint32_t b0 = (uint32_t)(L.w * MT * M::TB);
    const int bl = L.j / M::S, jj = L.j % M::S;
    {
        const uint32_t* sp = src.p0 + L.w * MT * 256 + pos;
        uint4 x[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) x[t] = ld4(sp + t * 256);
        for (int k = 1; k < src.n; ++k)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const uint4 e = ld4(sp + k * src.stride + t * 256);
                x[t].x = addm(x[t].x, e.x, P.p), x[t].y = addm(x[t].y, e.y, P.p);
                x[t].z = addm(x[t].z, e.z, P.p), x[t].w = addm(x[t].w, e.w, P.p);
            }
        MfMat X, Y;
        MfInit<false> cx, cy;
        Y.load(T, pid, MF_INV + MF_Y2, L.lane);
        cy.template load<M::S>(T, pid, MF_INV + MF_Y2, L.lane);
        X.load(T, pid, MF_INV + MF_X16, L.lane);
        cx.template load<16>(T, pid, MF_INV + MF_X16, L.lane);
        const uint4 xi = ld4(tw + M::XI + pos % M::C);
        uint32_t* l = lds + L.w * MT * 256;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            uint32_t y[4] = {x[t].x, x[t].y, x[t].z, x[t].w};
            mf_apply(y, Y, cy, P);
            mf_twist(y, xi, P);
            mf_twist(y, ld4(tw + M::TWB + (b0 + t * M::TB + pos / M::C) * 16 + 4 * L.q), P);
            *(uint4*)(l + t * 256 + mf_pos(pos)) = make_uint4(y[0], y[1], y[2], y[3]);
        }
        wave_sync();
        uint32_t z[MT][4];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) z[t][v] = l[t * 256 + mf_pos(bl * M::C + (4 * v + L.q) * M::S + jj)];
        wave_sync();
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            mf_apply(z[t], X, cx, P);
            mf_twist(z[t], ld4(tw + M::TW2 + (b0 + t * M::TB + bl) * 16 + 4 * L.q), P);
#pragma unroll
            for (int m = 0; m < 4; ++m) lds[O::pos(b0 + t * M::TB + bl, (4 * m + L.q) * M::S + jj)] = z[t][m];
        }
    }
    MfMat X, Y;
    MfInit<true> cx;
    MfInit<false> cy;
    Y.load(T, pid, MF_INV + MF_Y1, L.lane);
    cy.template load<M::T1>(T, pid, MF_INV + MF_Y1, L.lane);
    X.load(T, pid, MF_INV + MF_X1, L.lane);
    cx.template load<16>(T, pid, MF_INV + MF_X1, L.lane);
    const uint32_t s = A.es ? sload((const uint32_t*)A.es + i) : sload((const uint32_t*)A.ninv + pid);
    const uint32_t ss = A.es ? sload((const uint32_t*)A.ess + i) : sload((const uint32_t*)A.ninvs + pid);
    const uint32_t tau = (uint32_t)(L.w * MT % M::T1), col = (uint32_t)(L.w * MT / M::T1 * 16 + L.j);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const uint32_t r = 16 * (tau + t) + 4 * L.q;
        uint32_t y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = lds[O::pos(r + v, col)];
        mf_apply(y, Y, cy, P);
        mf_twist(y, ld4(tw + M::TW1 + r), P);
#pragma unroll
        for (int m = 0; m < 4; ++m) lds[O::pos(r + m, col)] = y[m];
    }
    __syncthreads();
    const Buf bo((const uint32_t*)A.base + (row_off(A, i) << LOGN), (uint32_t)M::N * 4);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        uint32_t y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = lds[O::pos(tau + t + M::T1 * (4 * v + L.q), col)];
        mf_apply(y, X, cx, P);
#pragma unroll
        for (int m = 0; m < 4; ++m)
            bo.st(shoup(y[m], s, ss, P.p), ((tau + M::T1 * L.q) * M::C + col) * 4,
                  (uint32_t)((t + M::T1 * 4 * m) * M::C) * 4);
    }
}

// ------------------------------------------------------------------------------------------------ launchers
inline int mf_check(const NttArgs* a, const MfTab* t, bool fwd) {
    if (!a || !t || a->nrows < 0 || !a->base || !a->roff || !a->rprime || !a->pr) return -1;
    if (!t->tw || !t->itw || !t->mat || !t->init || t->can < 1) return -1;
    if (a->soff && (!a->src || a->snum < 1 || (fwd && a->snum != 1))) return -1;
    if (fwd && a->epi != 0) {
        if (a->epi < 1 || a->epi > 3 || !a->eout || !a->ex || !a->es || !a->ess || a->xnum < 1) return -2;
    } else if (a->epi != 0) {
        return -2;
    }
    if (!fwd && !a->es && (!a->ninv || !a->ninvs)) return -1;
    return 0;
}
// whether a whole transform of rows of N takes the one-pass form
template <int LOGN>
bool mf_one(int rows) { return rows > 0 && (LOGN <= 13 || one14(rows)); }
template <int LOGN, int CAN>
void mf_one_launch(const NttArgs& A, const MfTab& T, const RescaleArgs* R, hipStream_t st) {
    const dim3 g(A.nrows), b(64 * Mo<LOGN>::W);
    if (R) {
        hipLaunchKernelGGL((mf_fwd_one<LOGN, 3, CAN, true>), g, b, 0, st, A, T, *R);
        return;
    }
    switch (A.epi) {
        case 0: hipLaunchKernelGGL((mf_fwd_one<LOGN, 0, CAN>), g, b, 0, st, A, T, RescaleArgs{}); break;
        case 1: hipLaunchKernelGGL((mf_fwd_one<LOGN, 1, CAN>), g, b, 0, st, A, T, RescaleArgs{}); break;
        case 2: hipLaunchKernelGGL((mf_fwd_one<LOGN, 2, CAN>), g, b, 0, st, A, T, RescaleArgs{}); break;
        default: hipLaunchKernelGGL((mf_fwd_one<LOGN, 3, CAN>), g, b, 0, st, A, T, RescaleArgs{}); break;
    }
}
template <int LOGN, int CAN>
void mf_rows_launch(const NttArgs& B, const MfTab& T, int r0, int n, hipStream_t st) {
    const dim3 g(Mg<LOGN>::N / Mg<LOGN>::LDS, n), b(64 * MW);
    switch (B.epi) {
        case 0: hipLaunchKernelGGL((mf_fwd_rows<LOGN, 0, CAN>), g, b, 0, st, B, T, r0); break;
        case 1: hipLaunchKernelGGL((mf_fwd_rows<LOGN, 1, CAN>), g, b, 0, st, B, T, r0); break;
        case 2: hipLaunchKernelGGL((mf_fwd_rows<LOGN, 2, CAN>), g, b, 0, st, B, T, r0); break;
        default: hipLaunchKernelGGL((mf_fwd_rows<LOGN, 3, CAN>), g, b, 0, st, B, T, r0); break;
    }
}
// cols: both passes, else the row pass alone; R: the column pass generates rescale corrections
template <int LOGN>
int mf_fwd(const NttArgs* a, const MfTab* t, pc_stream_t s, bool cols, const RescaleArgs* R = nullptr) {
    if (int rc = mf_check(a, t, true)) return rc;
    if (R && a->soff) return -1;
    using M = Mg<LOGN>;
    const NttArgs A = *a;
    if constexpr (LOGN <= 14) {
        if (cols && (!R || A.epi == 3) && mf_one<LOGN>(A.nrows)) {
            if (t->can == 1) mf_one_launch<LOGN, 1>(A, *t, R, (hipStream_t)s);
            else mf_one_launch<LOGN, 2>(A, *t, R, (hipStream_t)s);
            return launch_rc();
        }
    }
    const int chunk = A.chunk > 0 && cols ? A.chunk : (A.nrows > 0 ? A.nrows : 1);
    hipStream_t st = (hipStream_t)s;
    for (int r0 = 0; r0 < A.nrows; r0 += chunk) {
        const int n = A.nrows - r0 < chunk ? A.nrows - r0 : chunk;
        const dim3 g(M::C / M::COLS, n), b(64 * MW);
        if (R) hipLaunchKernelGGL((mf_fwd_cols<LOGN, true>), g, b, 0, st, A, *t, r0, *R);
        else if (cols) hipLaunchKernelGGL((mf_fwd_cols<LOGN>), g, b, 0, st, A, *t, r0, RescaleArgs{});
        NttArgs B = A;
        B.soff = nullptr;
        if (t->can == 1) mf_rows_launch<LOGN, 1>(B, *t, r0, n, st);
        else mf_rows_launch<LOGN, 2>(B, *t, r0, n, st);
    }
    return launch_rc();
}
template <int LOGN>
int mf_inv(const NttArgs* a, const MfTab* t, pc_stream_t s) {
    if (int rc = mf_check(a, t, false)) return rc;
    using M = Mg<LOGN>;
    const NttArgs A = *a;
    if constexpr (LOGN <= 14) {
        if (mf_one<LOGN>(A.nrows)) {
            hipLaunchKernelGGL((mf_inv_one<LOGN>), dim3(A.nrows), dim3(64 * Mo<LOGN>::W), 0, (hipStream_t)s, A, *t);
            return launch_rc();
        }
    }
    const int chunk = A.chunk > 0 ? A.chunk : (A.nrows > 0 ? A.nrows : 1);
    hipStream_t st = (hipStream_t)s;
    for (int r0 = 0; r0 < A.nrows; r0 += chunk) {
        const int n = A.nrows - r0 < chunk ? A.nrows - r0 : chunk;
        hipLaunchKernelGGL((mf_inv_rows<LOGN>), dim3(M::N / M::LDS, n), dim3(64 * MW), 0, st, A, *t, r0);
        NttArgs B = A;
        B.soff = nullptr;
        hipLaunchKernelGGL((mf_inv_cols<LOGN>), dim3(M::C / M::COLS, n), dim3(64 * MW), 0, st, B, *t, r0);
    }
    return launch_rc();
}

// ------------------------------------------------------------------------------------------------ tables
// Entry e of prime blockIdx.y's table (TW1 | TW2 | TWB | XI): the power of its root, times 2^32
__global__ void __launch_bounds__(256) mf_tw_k(int logn, const uint32_t* fw, const PrimeConst* pr, uint32_t* tw) {
    const int lr = logn / 2, lc = logn - lr;
    const uint32_t twn = mf_tw_words(logn), R = 1u << lr, e = blockIdx.x * 256 + threadIdx.x, id = blockIdx.y;
    if (e >= twn) return;
    const uint32_t rho1 = R / 16, rho2 = 1u << (lc - 4);
    uint32_t x, k;  // the root as an index of fw, the power
    if (e < R) {  // level 16, radix R / 16, by position
        x = rho1 / 2 * (16 + e / rho1), k = e % rho1;
    } else if (e < 17 * R) {  // level R, radix 16, [block][quarter][v]: k = q + 4 v
        const uint32_t f = e - R;
        x = 8 * (R + f / 16), k = ((f >> 2) & 3) + 4 * (f & 3);
    } else if (e < 33 * R) {  // level 16 R, radix C / 16: beta of block f / 16
        const uint32_t f = e - 17 * R;
        x = rho2 / 2 * 16 * (R + f / 16), k = f % 16 % rho2;
    } else {  // xi of child f / rho2: fw[i] = psi^brev(i) for every i, also below a level's first entry
        const uint32_t f = e - 33 * R;
        x = rho2 / 2 * (f / rho2), k = f % rho2;
    }
    const Red red(pr[id]);
    uint32_t b = fw[((size_t)id << logn) + x], v = red.r32;
    for (; k; k >>= 1) {
        if (k & 1) v = red.mul(v, b);
        b = red.mul(b, b);
    }
    tw[(size_t)id * twn + e] = v;
}

}  // namespace ntt

int mf_build_tw(int logn, int ids, const uint32_t* fw, const uint32_t* iw, const PrimeConst* pr, uint32_t* tw,
                uint32_t* itw, pc_stream_t s) {
    if (logn < 12 || logn > 16 || ids < 1 || !fw || !iw || !pr || !tw || !itw) return -1;
    const dim3 g((mf_tw_words(logn) + 255) / 256, ids);
    hipLaunchKernelGGL(ntt::mf_tw_k, g, dim3(256), 0, (hipStream_t)s, logn, fw, pr, tw);
    hipLaunchKernelGGL(ntt::mf_tw_k, g, dim3(256), 0, (hipStream_t)s, logn, iw, pr, itw);
    return launch_rc();
}

int mf_can(const uint64_t* primes, int n) {
    // a step's word is below 1.13 p + lo, lo <= (2^21 + 255) 257
    const double lo = 2097407.0 * 257.0;
    int can = 1;
    for (int i = 0; i < n; ++i) {
        const double r = 1.13 * (double)primes[i] + lo;
        if (r >= 4.0 * (double)primes[i]) return 0;
        if (r >= 2.0 * (double)primes[i]) can = 2;
    }
    return can;
}

namespace {
uint64_t mulm(uint64_t a, uint64_t b, uint64_t p) { return a * b % p; }  // p < 2^31
uint64_t powm(uint64_t b, uint64_t e, uint64_t p) {
    uint64_t r = 1 % p;
    for (; e; e >>= 1, b = mulm(b, b, p))
        if (e & 1) r = mulm(r, b, p);
    return r;
}
uint32_t brev_h(uint32_t x, int bits) {
    uint32_t r = 0;
    for (int i = 0; i < bits; ++i) r |= ((x >> i) & 1u) << (bits - 1 - i);
    return r;
}
}  // namespace

void mf_digits(uint64_t w, uint64_t p, int8_t (&d)[4]) {
    int64_t v = w > p / 2 ? (int64_t)w - (int64_t)p : (int64_t)w;
    for (int i = 0; i < 4; ++i) {
        d[i] = (int8_t)(uint8_t)(v & 255);
        v = (v - d[i]) >> 8;
    }
}

void mf_build_mats(int logn, uint64_t p, uint64_t psi, uint32_t* mat, uint32_t* init) {
    const uint64_t n = 1ull << logn;
    const int lr = logn / 2, lc = logn - lr;
    const uint64_t ipsi = powm(psi, 2 * n - 1, p);
    for (int which = 0; which < MF_MATS; ++which) {
        const bool inv = which >= MF_INV;
        const int kind = which % MF_INV;
        const int lrho = kind == MF_Y1 ? lr - 4 : kind == MF_Y2 ? lc - 4 : 4;
        const uint32_t rho = 1u << lrho;
        const uint64_t root = inv ? ipsi : psi;
        // F[o][k]: forward o the child c and k the word; inverse o the word and k the child
        uint64_t F[16][16];
        for (uint32_t o = 0; o < 16; ++o)
            for (uint32_t k = 0; k < 16; ++k) {
                const uint32_t c = (inv ? k : o) % rho, w = (inv ? o : k) % rho;
                if (o / rho != k / rho) {
                    F[o][k] = 0;
                    continue;
                }
                uint64_t e = (uint64_t)w * brev_h(c, lrho) % rho * (2 * n / rho);  // omega^(w brev(c))
                if (kind == MF_X1) e += (uint64_t)w * (n / 16);  // eta = fw[8] = psi^(brev(8)) = psi^(N / 16)
                F[o][k] = powm(root, e, p);
            }
        const bool x = kind == MF_X1 || kind == MF_X16;  // k = q + 4 v, o = 4 m + q; else k = 4 q + v, o = 4 q + m
        std::vector<int8_t> bytes(4096);
        for (int m = 0; m < 4; ++m)
            for (int lane = 0; lane < 64; ++lane) {
                const int row = lane % 16, qo = row / 4, dig = row % 4, ql = lane / 16;
                const int o = x ? 4 * m + qo : 4 * qo + m;
                for (int v = 0; v < 4; ++v) {
                    const int k = x ? ql + 4 * v : 4 * ql + v;
                    for (int a = 0; a < 4; ++a) {
                        int8_t d[4];
                        mf_digits(mulm(F[o][k], (1ull << (8 * a)) % p, p), p, d);
                        bytes[((m * 64 + lane) * 4 + v) * 4 + a] = d[dig];
                    }
                }
            }
        memcpy(mat + which * 1024, bytes.data(), 4096);
        // sum_i c_i 2^(8i) == 128 sum_{k,a} W (mod p) with c_i = 2^20 + d_i >= the largest |sum| of a digit's products
        const uint64_t B = 1u << 20, ones = 0x01010101ull;
        for (int m = 0; m < 4; ++m)
            for (int q = 0; q < 4; ++q) {
                const int o = x ? 4 * m + q : 4 * q + m;
                uint64_t s = 0;
                for (int k = 0; k < 16; ++k) s = (s + mulm(F[o][k], ones % p, p)) % p;
                const uint64_t need = (mulm(s, 128, p) + p - mulm(B % p, ones % p, p)) % p;
                for (int i = 0; i < 4; ++i)
                    init[which * 64 + (m * 4 + q) * 4 + i] = (uint32_t)(B + ((need >> (8 * i)) & 255));
            }
    }
}

#define PCH_MF(CALL)                 \
    switch (logn) {                  \
        case 12: return ntt::CALL(12); \
        case 13: return ntt::CALL(13); \
        case 14: return ntt::CALL(14); \
        case 15: return ntt::CALL(15); \
        case 16: return ntt::CALL(16); \
        default: return -2;          \
    }
int mf_ntt_fwd(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s) {
#define PCH_C(L) mf_fwd<L>(a, t, s, true)
    PCH_MF(PCH_C)
#undef PCH_C
}
int mf_ntt_fwd_rows(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s) {
#define PCH_C(L) mf_fwd<L>(a, t, s, false)
    PCH_MF(PCH_C)
#undef PCH_C
}
int mf_ntt_fwd_rescale(int logn, const NttArgs* a, const RescaleArgs* r, const MfTab* t, pc_stream_t s) {
#define PCH_C(L) mf_fwd<L>(a, t, s, true, r)
    PCH_MF(PCH_C)
#undef PCH_C
}
int mf_ntt_inv(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s) {
#define PCH_C(L) mf_inv<L>(a, t, s)
    PCH_MF(PCH_C)
#undef PCH_C
}

}  // namespace pch
