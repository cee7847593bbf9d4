// Transforms on the matrix cores: the tables and device building blocks of the MFMA NTT passes (mfntt.hip) and of the
// passes that fuse a base conversion into them.
//
// A modular product of a vector of 16 words by a fixed 16 x 16 matrix F over a prime p is one int8 contraction of depth
// 64 per output digit. A word x is its four bytes b_a; sum_k F[o][k] x_k = sum_{k,a} (F[o][k] 2^(8a) mod p) b_a(x_k),
// and each multiplier W = F 2^(8a) mod p (centred, |W| < 2^30) is four signed base-256 digits W = sum_i w_i 2^(8i). So
// S_i = sum_{k,a} w_i b_a gives the output as sum_i S_i 2^(8i) mod p: v_mfma_i32_16x16x64_i8 forms, for 16 vectors, the
// four S_i of four outputs. The bytes enter as b - 128 (the word xor 0x80808080), so that they are signed; the constant
// 128 sum W and a bias that keeps every S_i non-negative are the accumulator's initial value. With |b - 128| and |w|
// at most 128, |sum| <= 64 2^14 = 2^20, so S_i < 2^21 + 2^8 and the value is below 2^46: one quotient estimate reduces
// it to r < 1.13 p + 2^29.01 (mf_reduce). The words between steps are any 32-bit words, so no step needs a correction.
// A conversion of 17 to 20 sources has depth 80: |sum| <= 80 2^14 = 1.25 2^20 under a bias of 2^21, so S_i < 3.25 2^20 + 2^8,
// S_2 + S_3 2^8 and S_0 + S_1 2^8 are below 257 (3.25 2^20 + 2^8) < 2^29.71, and the estimate is low by less than 1 +
// 2^29.71 / 2^32 < 1.21: r < 1.21 p + 2^29.71, below 2^32 for p < 2^31.
//
// A radix-rho step of the transform at a level of m blocks takes block i's words x_k (k < rho, N / (rho m) apart) to
// their values at the rho roots: out_c = sum_k (x_k eta^k) omega^(k brev(c)), eta = fw[(rho / 2)(m + i)], omega =
// psi^(2N / rho): a product per word by a power of eta, then the matrix omega^(k brev(c)), the same for every block of
// every level (rho = 8 and 4: two or four small matrices on the diagonal of the 16 x 16 one). At the first level there
// is one block and eta^k is folded into the matrix. The inverse step is the transposed pair: the matrix
// omega^(-k brev(c)), then the product by eta^(-k). The twiddles are in Montgomery form (w 2^32 mod p): a product is
// three instructions, as Shoup's, with one table word instead of two (mf_mont).
//
// A row pass's second step has a block per 16 words, N twiddles in all; brev is linear over disjoint bits, so they
// factor: child c of the pass's block b has eta = beta_b xi_c, beta_b = fw[(C / 2)(R + b)] and xi_c = psi^brev((C / 32) c).
// xi_c^k is the same C words for every block, held in registers, and beta_b^k 16 words per block: two products per word
// instead of N table words read beside N data words.
//
// A radix-16 step costs a word 9 VALU instructions (3 twiddle, 1 xor, 5 reduction; 12 with both factors) where its four
// butterfly stages cost 18 (14 below 2^30).
#pragma once
#include "common.h"

namespace pch {

// per context, by prime id (`rows` ids)
struct MfTab {
    const uint32_t* tw;    // forward twiddles (Montgomery form): [id][mf_tw_words]: TW1 | TW2 | TWB | XI
    const uint32_t* itw;   // their inverses, the same layout
    const uint32_t* mat;   // [id][MF_MATS][1024]: the matrices' digits in the MFMA A operand's lane order
    const uint32_t* init;  // [id][MF_MATS][64]: the accumulators' initial values [m][quarter][digit]
    int can;               // final corrections of a transform's words: 1 or 2 (mf_can)
};
// the matrices: X1 (first level, eta folded in), X16 (omega_16), Y1 (a column pass's second radix), Y2 (a row pass's);
// then their inverses
enum { MF_X1 = 0, MF_X16 = 1, MF_Y1 = 2, MF_Y2 = 3, MF_INV = 4, MF_MATS = 8 };
// the twiddles: TW1, the column pass's second step by row position (R words); TW2, the row pass's first step by block,
// [quarter][v] (16 R); TWB, its second step's beta_b^k by block, 4 quarter + v (16 R); XI, xi_c^k by word of the block (C)
constexpr uint32_t mf_tw_words(int logn) { return (33u << (logn / 2)) + (1u << (logn - logn / 2)); }

#if defined(__HIP_DEVICE_COMPILE__) || defined(__HIPCC__)
typedef int v4i __attribute__((ext_vector_type(4)));
constexpr uint32_t MF_FLIP = 0x80808080u;

struct MfPrime {
    uint32_t p, np, mu, pinv;  // p, 2^32 - p, floor(2^48 / p), -p^-1 mod 2^32
    __device__ __forceinline__ MfPrime(uint32_t p_, uint32_t mu_, uint32_t pinv_)
        : p(p_), np(0u - p_), mu(mu_), pinv(pinv_) {}
    __device__ __forceinline__ MfPrime(const PrimeConst* pr, uint32_t i) {
        p = (uint32_t)sload(&pr[i].p);
        np = 0u - p;
        mu = (uint32_t)(sload(&pr[i].mu_lo) >> 16);
        pinv = (uint32_t)sload(&pr[i].mont_pinv);
    }
};

// S_0 + S_1 2^8 + S_2 2^16 + S_3 2^24 as a word r == it (mod p), at depth 64. With hi = S_2 + S_3 2^8 < 2^29.01, the quotient q =
// floor(hi mu / 2^32) of hi 2^16 by p is low by less than 1.13, so hi 2^16 - q p < 1.13 p and r < 1.13 p + lo, lo < 2^29.01:
// below 2^32 for every p < 2^31.
template <int SH>
__device__ __forceinline__ uint32_t lshl_add(uint32_t a, uint32_t b) {  // (a << SH) + b, kept as one instruction
    uint32_t d;
    asm("v_lshl_add_u32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "n"(SH), "v"(b));
    return d;
}
__device__ __forceinline__ uint32_t mf_reduce(const v4i& s, const MfPrime& P) {
    // the first readers of the MFMA's registers are instructions that the compiler emits (and separates from the MFMA by
    // the wait states it owes), never inline assembly
    const uint32_t lo = ((uint32_t)s.y << 8) + (uint32_t)s.x, hi = ((uint32_t)s.w << 8) + (uint32_t)s.z;
    const uint32_t q = __umulhi(hi, P.mu);
    const uint32_t t = lshl_add<16>(hi, lo);
    uint64_t r, c;
    const uint64_t a = ((uint64_t)hi << 32) | t;  // only the low word matters: hi is there so that no register is cleared
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(c) : "v"(q), "s"(P.np), "v"(a));
    return (uint32_t)r;
}
// a w 2^-32 mod p in [0, 2p) for any word a and w < p: a w + m p with m = a w pinv mod 2^32 is a multiple of 2^32 below
// 2^33 p
__device__ __forceinline__ uint32_t mf_mont(uint32_t a, uint32_t w, const MfPrime& P) {
    uint64_t aw, r, c0, c1;
    asm("v_mad_u64_u32 %0, %1, %2, %3, 0" : "=v"(aw), "=s"(c0) : "v"(a), "v"(w));
    const uint32_t m = (uint32_t)aw * P.pinv;
    asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(c1) : "v"(m), "s"(P.p), "v"(aw));
    return (uint32_t)(r >> 32);
}
// a step's word as its residue: CAN conditional subtractions (mf_can)
template <int CAN>
__device__ __forceinline__ uint32_t mf_canon(uint32_t r, const MfPrime& P) {
    if (CAN == 2) r = min(r, r - 2 * P.p);
    return min(r, r - P.p);
}

// one matrix of a prime: the A operands of its four MFMAs (outputs 4 m + quarter or 4 quarter + m)
struct MfMat {
    v4i a[4];
    __device__ __forceinline__ void load(const MfTab& T, uint32_t id, int which, int lane) {
        const v4i* m = (const v4i*)(T.mat + ((size_t)id * MF_MATS + which) * 1024) + lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = m[64 * k];
    }
};
// the initial accumulators. An output's depends on the sum of its matrix row: zero for every output but those that sum
// the all-ones row (the matrix's or a diagonal block's output 0, all in MFMA 0); X1's (FULL) each have their own
template <bool FULL>
struct MfInit {
    v4i c[FULL ? 4 : 2];
    // RHO: the matrix's radix (FULL: unused)
    template <int RHO>
    __device__ __forceinline__ void load(const MfTab& T, uint32_t id, int which, int lane) {
        const uint32_t* t = T.init + ((size_t)id * MF_MATS + which) * 64;
        const int q = lane >> 4;
        if constexpr (FULL) {
#pragma unroll
            for (int k = 0; k < 4; ++k) c[k] = ((const v4i*)t)[4 * k + q];
        } else {
            const bool one = (4 * q) % RHO == 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int g = (int)sload(t + 16 + i), z = (int)sload(t + i);
                c[1][i] = g;
                c[0][i] = one ? z : g;
            }
        }
    }
    __device__ __forceinline__ const v4i& operator[](int m) const { return c[FULL ? m : (m ? 1 : 0)]; }
};
template <bool FULL>
__device__ __forceinline__ void mf_apply(uint32_t (&x)[4], const MfMat& M, const MfInit<FULL>& I, const MfPrime& P) {
    const v4i b = {(int)(x[0] ^ MF_FLIP), (int)(x[1] ^ MF_FLIP), (int)(x[2] ^ MF_FLIP), (int)(x[3] ^ MF_FLIP)};
    v4i d[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) d[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(M.a[m], b, I[m], 0, 0, 0);
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = mf_reduce(d[m], P);
}
__device__ __forceinline__ void mf_twist(uint32_t (&x)[4], const uint4& w, const MfPrime& P) {
    x[0] = mf_mont(x[0], w.x, P);
    x[1] = mf_mont(x[1], w.y, P);
    x[2] = mf_mont(x[2], w.z, P);
    x[3] = mf_mont(x[3], w.w, P);
}
#endif

// host: corrections that take a step's word (r < 1.13 p + 2^29.01) to its residue for every prime of the list: 1 where
// that is below 2p, 2 where it is below 4p, 0 where the matrix passes do not apply
int mf_can(const uint64_t* primes, int n);
// host: the twiddle tables by a kernel from the butterfly tables (device, [id][N]), into tw / itw
int mf_build_tw(int logn, int ids, const uint32_t* fw, const uint32_t* iw, const PrimeConst* pr, uint32_t* tw,
                uint32_t* itw, pc_stream_t s);
// host: the matrices and initial values of one prime (psi: its 2N-th root), MF_MATS x 1024 and MF_MATS x 64 words
void mf_build_mats(int logn, uint64_t p, uint64_t psi, uint32_t* mat, uint32_t* init);

// the table's ntt_fwd / ntt_inv on the matrix cores (the same NttArgs and epilogues; no dense launches)
int mf_ntt_fwd(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s);
int mf_ntt_inv(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s);
// the row pass alone, after a column pass done elsewhere
int mf_ntt_fwd_rows(int logn, const NttArgs* a, const MfTab* t, pc_stream_t s);
// A base-conversion plan on the matrix cores (mfconv.hip). Job k takes its source rows (src_off + a row, words prescaled;
// every word any 32 bits) to the column pass of its targets in rows dst_off + a row.
struct MfConvJob {
    uint32_t src_off, dst_off;    // rows
    uint32_t src_rows, dst_rows;  // the extents: rows read and written lie below them
    uint32_t nt;                  // targets
    uint32_t dig;                 // words of MfConvArgs.dig: mf_conv_digits of each four targets
    uint32_t pad[2];
};
struct MfConvTgt {
    uint32_t row, id, p, mu, pinv, pad[3];  // its row and prime id; MfPrime's constants
};
struct MfConvArgs {
    const uint32_t* src;
    uint32_t* dst;
    const uint32_t* jobs;  // job k's words from k stride: MfConvJob, src_words(ns) source rows (past the last: any of
    const uint32_t* dig;   // them), nt MfConvTgt
    uint32_t stride;
    int njobs, max_tgt, ns;  // ns: 8, 16 or 20, the jobs' sources padded
    static constexpr __host__ __device__ uint32_t src_words(int ns) { return ((uint32_t)ns + 7) / 8 * 8; }
    static constexpr __host__ __device__ uint32_t group_words(int ns) { return (uint32_t)ns * 16 + 16; }
};
constexpr int MFC_MAX_NS = 20;
// tpw: targets per workgroup: 1, 2 or a multiple of 4. 0, -1 (bad arguments), -2 (ns or logn outside the range) or a HIP error
int mf_conv_cols(int logn, const MfConvArgs* a, const MfTab* t, int tpw, pc_stream_t s);
// u = floor(sum_i y_i / b_i + 1/2) of each exact job of a (bconv.hip's records: the doubles' FMAs in source order) to row k
// of u, job k's
int conv_u(int logn, const BconvArgs* a, uint32_t* u, pc_stream_t s);
// host: the A operands and initial values of one run of nt <= 4 targets: w[i][t] below p[t], n sources padded to ns
void mf_conv_digits(const uint64_t* w, int n, int nt, const uint64_t* p, int ns, uint32_t* out);
// host: the four signed base-256 digits of w mod p, centred
void mf_digits(uint64_t w, uint64_t p, int8_t (&d)[4]);
// the table's rescale_fwd (rescale.hip) with its transform on the matrix cores
int mf_rescale_fwd(int logn, const RescaleNttArgs* a, const MfTab* t, pc_stream_t s);
// the forward transform of composite-rescale corrections (ntt_fwd_rescale)
int mf_ntt_fwd_rescale(int logn, const NttArgs* a, const RescaleArgs* r, const MfTab* t, pc_stream_t s);

}  // namespace pch
