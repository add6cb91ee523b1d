// chol.hip -- batched Cholesky factorisation / solve for gfx950.
//
// Replaces cusolverDn?potrfBatched / ?potrsBatched of GPUtils'
// CholeskyBatchFactoriser (include/tensor.cuh:2098-2197) and adds a fused
// factor+solve.  The mixed-precision solve (FP32 factor, FP64 refinement)
// is in chol_mixed.hip and n <= 32 in chol_small.hip; its C entry point is
// here, with this file's FP64 kernel as the fallback for systems that do
// not converge.
//
// Design (one 256-thread workgroup = 4 wavefronts per matrix):
//  * The lower block triangle of the matrix lives in LDS as 16x16 blocks
//    (block (I,J), I >= J, at index I(I+1)/2 + J, column-major inside the
//    block with the row index XOR-ed by the column, see sw()).  n is padded to a multiple of 16 with an identity tail, so the
//    padded factor is diag(L, I) and no kernel path needs edge masks.
//  * Right-looking blocked algorithm, per block column J:
//      1. wave 0 factors the 16x16 diagonal block in registers (one row per
//         lane, broadcasts through v_readlane) and forms its triangular
//         inverse D_J; D_J replaces L_JJ in LDS (L_JJ goes straight to HBM
//         when the factor is an output);
//      2. panel   L_IJ = A_IJ D_J^T      (16x16x4 MFMA, 4 per block);
//      3. update  A_IK -= L_IJ L_KJ^T    (16x16x4 MFMA, 4 per tile).
//    Both MFMA operands of a 16x16x4 step read element
//    (lane % 16, lane / 16 + 4 kk) of their block.
//  * Triangular solves use the same block inverses: per block row a 16x16
//    matrix-vector product replaces the serial substitution.
#include <mutex>
#include <type_traits>

#include "chol_mixed.hpp"
#include "chol_small.hpp"
#include "common.hpp"
#include "householder.hpp"

namespace gputils {
namespace chol {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kRhsChunk = 4;  // right-hand sides per solve sweep (lane = row + 16*rhs)

__host__ __device__ constexpr int tri(int I) { return (I * (I + 1)) >> 1; }

// Element (r, c) of a 16x16 block in LDS sits at sw(r, c): column-major with
// the row index XOR-ed by the column.  A column (fixed c) still fills 16
// consecutive slots, and a row (fixed r, c = 0..15), which the MFMA
// accumulator layout and the transposed solves read and write, falls in
// 16 different banks instead of one (a plain column-major 16x16 block of
// doubles puts a row on a 128-byte stride).
__device__ __forceinline__ int sw(int r, int c) { return (r ^ c) + 16 * c; }

// Load the lower triangle of the n x n matrix A (column-major, lda) into
// LDS block storage with identity padding up to 16*nb.  Thread t owns
// element (t % 16, t / 16) of every block; blocks are fetched eight at a
// time so that each thread keeps eight independent loads in flight.
template <typename Tin, typename T>
__device__ __forceinline__ void load_lower(const Tin *__restrict__ A, int64_t lda, int n, int nb, T *L) {
    const int i = threadIdx.x & 15, k = threadIdx.x >> 4;
    const int nblk = tri(nb);
    int I = 0, J = 0;  // coordinates of block b0 (uniform)
    for (int b0 = 0; b0 < nblk; b0 += 8) {
        T v[8];
        int Iu = I, Ju = J;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int gi = 16 * Iu + i, gk = 16 * Ju + k;
            T x = (gi == gk) ? T(1) : T(0);
            if (b0 + u < nblk && gi < n && gk < n && gi >= gk) x = (T)A[gi + (int64_t)gk * lda];
            v[u] = x;
            if (++Ju > Iu) { ++Iu; Ju = 0; }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (b0 + u < nblk) L[(b0 + u) * 256 + sw(i, k)] = v[u];
        I = Iu;
        J = Ju;
    }
}

// Store the strictly-below-diagonal blocks (I > J) back to A.
template <typename T>
__device__ __forceinline__ void store_offdiag(T *__restrict__ A, int64_t lda, int n, int nb, const T *L) {
    const int i = threadIdx.x & 15, k = threadIdx.x >> 4;
    for (int I = 1; I < nb; ++I) {
        const int gi = 16 * I + i;
        for (int J = 0; J < I; ++J) {
            const int gk = 16 * J + k;
            if (gi < n && gk < n) A[gi + (int64_t)gk * lda] = L[(tri(I) + J) * 256 + sw(i, k)];
        }
    }
}

// Pivot of column k: inv = 1/sqrt(d), and s = sqrt(d), for d > 0.  inv is on
// the critical path of every column, s is not.  FP32 uses the hardware
// reciprocal square root (v_rsq_f32, 1 ulp).  FP64 refines the hardware
// estimate r = v_rsq_f64: with e = 1 - d r^2 (one rounding of d r), one third
// order step inv = r + r e (1/2 + 3/8 e) leaves the estimate's error cubed
// (2^-22 or better becomes below 2^-63): inv is within 1 ulp and s, d inv with
// one Newton correction (d - s^2) inv / 2, is correctly rounded (60000
// pivots with estimate errors up to 2^-22 against exact arithmetic).  Five dependent
// operations behind the estimate instead of the eight of two coupled steps.
// Pivots below 2^-767 are scaled by 2^256 first, as the library square root
// does, to keep the estimate accurate.
__device__ __forceinline__ void pivot(float d, float &s, float &inv) {
    inv = __builtin_amdgcn_rsqf(d);
    s = d * inv;
}
__device__ __forceinline__ void pivot(double d, double &s, double &inv) {
    const bool tiny = d < 0x1p-767;
    const double dd = tiny ? d * 0x1p+256 : d;
    const double r = __builtin_amdgcn_rsq(dd);
    const double e = __builtin_fma(-(dd * r), r, 1.0);
    const double q = __builtin_fma(r * e, __builtin_fma(0.375, e, 0.5), r);
    double g = dd * q;
    g = __builtin_fma(__builtin_fma(-g, g, dd), 0.5 * q, g);
    s = tiny ? g * 0x1p-128 : g;
    inv = tiny ? q * 0x1p+128 : q;
}

// The same for every positive d: v_rsq_f32 takes a subnormal d for zero, and for
// an infinite one (a variable fixed by a penalty) s is infinite and inv zero,
// where the steps above make NaNs.
__device__ __forceinline__ void pivot_any(float d, float &s, float &inv) {
    const bool tiny = d < 0x1p-126f;
    const float dd = tiny ? d * 0x1p+48f : d;
    const float q = __builtin_amdgcn_rsqf(dd);  // 0 for infinity
    inv = tiny ? q * 0x1p+24f : q;
    s = __builtin_isinf(d) ? d : (tiny ? dd * q * 0x1p-24f : d * inv);
}
__device__ __forceinline__ void pivot_any(double d, double &s, double &inv) {
    pivot(d, s, inv);
    const bool inf = __builtin_isinf(d);
    inv = inf ? 0.0 : inv;
    s = inf ? d : s;
}

// d += (v of lane LANE of the 16-lane row) * w: the FMA takes the other
// lane's value by DPP (row_newbcast, the control that 64-bit arithmetic
// takes), where readlane and an FMA would be three instructions in FP64.
// The compiler does not form it by itself and does not see the hazards
// inside, so every group of them starts with the two wait states that a DPP
// source needs after a VALU write and ends with the one that a readlane of
// its result needs.
template <int LANE>
__device__ __forceinline__ void fma_lane(double &d, double v, double w) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\ts_nop 0" : "+v"(d) : "v"(v), "v"(w), "n"(LANE));
}
// FP32 is faster with readlane: two instructions, no wait states
// (v_fmac_f32_dpp made a 16x16 block 4096 cycles instead of 3701).
template <int LANE>
__device__ __forceinline__ void fma_lane(float &d, float v, float w) {
    d = fmaf(readlane(v, LANE), w, d);
}
// d_i += (v of lane LANE + i) * w, i < 4
template <int LANE>
__device__ __forceinline__ void fma_lanes4(double &d0, double &d1, double &d2, double &d3, double v, double w) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\ts_nop 0"
        : "+v"(d0), "+v"(d1), "+v"(d2), "+v"(d3)
        : "v"(v), "v"(w), "n"(LANE), "n"(LANE + 1), "n"(LANE + 2), "n"(LANE + 3));
}
template <int LANE>
__device__ __forceinline__ void fma_lanes4(float &d0, float &d1, float &d2, float &d3, float v, float w) {
    fma_lane<LANE>(d0, v, w);
    fma_lane<LANE + 1>(d1, v, w);
    fma_lane<LANE + 2>(d2, v, w);
    fma_lane<LANE + 3>(d3, v, w);
}
// acc0, acc1 += v_p(lane LANE) w_p for p, p + 1, p + 2, p + 3 (two chains)
template <int LANE, typename T>
__device__ __forceinline__ void dot_lane4(T &acc0, T &acc1, T v0, T v1, T v2, T v3, T w0, T w1, T w2, T w3) {
    if constexpr (sizeof(T) == 8)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %2, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %3, %7 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %0, %4, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %5, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
            : "+v"(acc0), "+v"(acc1)
            : "v"(v0), "v"(v1), "v"(v2), "v"(v3), "v"(w0), "v"(w1), "v"(w2), "v"(w3), "n"(LANE));
    else {
        fma_lane<LANE>(acc0, v0, w0);
        fma_lane<LANE>(acc1, v1, w1);
        fma_lane<LANE>(acc0, v2, w2);
        fma_lane<LANE>(acc1, v3, w3);
    }
}

// Row K of L^{-1} (lane c holding column c), without the division by the
// diagonal: e_K - sum_{p<K} L(K, p) x[p], from nx[p] = -x[p]; row[] holds
// the rows of L, lane r its row r, in every 16-lane row.
template <int K, typename T>
__device__ __forceinline__ T inverse_row(const T (&row)[16], const T (&nx)[16]) {
    T a0 = ((int)(threadIdx.x & 15) == K) ? T(1) : T(0), a1 = T(0);
    constexpr int K4 = K & ~3;
#pragma unroll
    for (int p = 0; p < K4; p += 4)
        dot_lane4<K>(a0, a1, row[p], row[p + 1], row[p + 2], row[p + 3], nx[p], nx[p + 1], nx[p + 2], nx[p + 3]);
#pragma unroll
    for (int p = K4; p < K; ++p) {
        if (p & 1) fma_lane<K>(a1, row[p], nx[p]);
        else fma_lane<K>(a0, row[p], nx[p]);
    }
    return a0 + a1;
}

// Steps K.. of the inversion of a lower triangular L (row[] as above), dinv
// the reciprocal of the lane's own diagonal entry: nx[K] = -row K of L^{-1}.
template <int K, typename T>
__device__ __forceinline__ void tri_inverse_steps(const T (&row)[16], T dinv, T (&nx)[16]) {
    if constexpr (K < 16) {
        nx[K] = -inverse_row<K>(row, nx) * readlane(dinv, K);
        asm volatile("" : "+v"(nx[K]));  // as in factor_steps
        tri_inverse_steps<K + 1>(row, dinv, nx);
    }
}

// Whether d is not a positive normal number: 1 or 0 from its bits, as d is
// uniform and the scalar unit has time beside the pivots' chain.
__device__ __forceinline__ unsigned unusual(float d) {
    return (unsigned)__float_as_int(d) - 0x00800000u >= 0x7f000000u;
}
__device__ __forceinline__ unsigned unusual(double d) {
    return (unsigned)(__double_as_longlong(d) >> 32) - 0x00100000u >= 0x7fe00000u;
}

// Steps K.. of the factorisation of a 16x16 block (see factor_diag_block).
// PIV: kNormal and kAny take pivot or pivot_any and leave the first failing
// step in `fail`; kWatch takes pivot and leaves whether a d was unusual.
constexpr int kNormal = 0, kAny = 1, kWatch = 2;
template <int PIV, int K, typename T>
__device__ __forceinline__ void factor_steps(T (&row)[16], T (&nx)[16], int lane, int &fail) {
    if constexpr (K < 16) {
        const T d = readlane(row[K], K);
        if constexpr (PIV == kWatch) fail |= unusual(d);
        else if (fail < 0 && !(d > T(0))) fail = K;  // uniform; also catches NaN
        T sq, inv;
        if constexpr (PIV == kAny) pivot_any(d, sq, inv);
        else pivot(d, sq, inv);
        const T lk = ((lane & 15) == K) ? sq : row[K] * inv;
        row[K] = lk;
        const T nl = -lk;
        constexpr int J4 = K + 1 + ((15 - K) & 3);  // the first 0..3 columns singly, the rest by fours
        if constexpr (K < 15) {
            if constexpr (J4 > K + 1) fma_lane<K + 1>(row[K + 1], lk, nl);
            if constexpr (J4 > K + 2) fma_lane<K + 2>(row[K + 2], lk, nl);
            if constexpr (J4 > K + 3) fma_lane<K + 3>(row[K + 3], lk, nl);
            if constexpr (J4 < 16) fma_lanes4<J4>(row[J4], row[J4 + 1], row[J4 + 2], row[J4 + 3], lk, nl);
            if constexpr (J4 + 4 < 16) fma_lanes4<J4 + 4>(row[J4 + 4], row[J4 + 5], row[J4 + 6], row[J4 + 7], lk, nl);
            if constexpr (J4 + 8 < 16) fma_lanes4<J4 + 8>(row[J4 + 8], row[J4 + 9], row[J4 + 10], row[J4 + 11], lk, nl);
        }
        nx[K] = -inverse_row<K>(row, nx) * inv;
        // left to the compiler, every row's readlane results were hoisted
        // into SGPRs and spilled
        asm volatile("" : "+v"(nx[K]));
        factor_steps<PIV, K + 1>(row, nx, lane, fail);
    }
}

// Factor the 16x16 diagonal block `blk` (lower part valid) with one
// wavefront and write D = L^{-1} over it (column-major).  If Lout != nullptr
// the factor L itself is written there (rows/cols < nvalid).
// Returns the index (0..15) of the first non-positive pivot or -1.
//
// Lane r < 16 holds row r (the other 16-lane rows repeat it).  Step k
// scales column k, applies its rank-1 update to the columns right of it and
// forms row k of L^{-1} (lane c holding column c), whose inputs -- row k of
// L -- are final at that point.  What bounds it is one wavefront's chain of
// pivots and its 240 FMAs, each taking its broadcast operand by DPP (about
// 9 cycles each; readlane and FMA: 12).  2048 FP64 systems of n = 128:
// factorisation 213 -> 205 us, solve (whose inverses now divide once per
// block instead of once per row) 99 -> 92 us, both fused 274 -> 260 us.  The 16 steps
// have no branch between them (a failed pivot is only recorded; the NaNs it
// spreads are never stored), so the pivot chain of column k + 1 overlaps
// the rest of step k.  Entries above the diagonal are updated with garbage
// and never read: only lanes r > j read row[j].
// ANY: pivots of the whole range of the type, for n > 128.  The 16 steps are
// done again with pivot_any where one was not a positive normal number (with it
// in all of them a block would take 20 % longer in FP32).
template <bool ANY = false, typename T>
__device__ __forceinline__ int factor_diag_block(T *blk, T *Lout, int64_t ldo, int nvalid) {
    // a lane index the compiler cannot relate to the one of the other
    // phases, so the per-step lane masks below are formed where they are
    // used instead of being kept live in SGPRs across the kernel
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    T row[16], nx[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) row[c] = blk[sw(lane & 15, c)];
    int fail = -1;
    if constexpr (ANY) {
        int odd = 0;
        factor_steps<kWatch, 0>(row, nx, lane, odd);
        if (__builtin_expect(odd, 0)) {
#pragma unroll
            for (int c = 0; c < 16; ++c) row[c] = blk[sw(lane & 15, c)];
            factor_steps<kAny, 0>(row, nx, lane, fail);
        }
    } else {
        factor_steps<kNormal, 0>(row, nx, lane, fail);
    }
    if (fail >= 0) return fail;
    if (Lout != nullptr && lane < 16 && lane < nvalid) {  // the rows below belong to others
#pragma unroll
        for (int c = 0; c < 16; ++c)
            if (c <= lane && c < nvalid) Lout[lane + (int64_t)c * ldo] = row[c];
    }
    if (lane < 16) {
#pragma unroll
        for (int r = 0; r < 16; ++r) blk[sw(r, lane)] = -nx[r];
    }
    return -1;
}

// C -= A_op * B_op^T for one 16x16 tile (all operands 16x16 LDS blocks,
// column-major); two tiles are interleaved for MFMA latency hiding.
template <typename T>
__device__ __forceinline__ void tile_update2(T *c0, const T *a0, const T *b0, T *c1, const T *a1,
                                    const T *b1, bool two) {
    using M = Mfma16<T>;
    const int lane = threadIdx.x & 63;
    const int col = lane & 15;
    typename M::acc_t x0, x1;
#pragma unroll
    for (int r = 0; r < 4; ++r) x0[r] = c0[sw(M::drow(lane, r), col)];
    if (two) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x1[r] = c1[sw(M::drow(lane, r), col)];
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const int o = sw(col, (lane >> 4) + 4 * kk);  // operand element (lane % 16, lane / 16 + 4 kk)
        x0 = M::fma(-a0[o], b0[o], x0);
        if (two) x1 = M::fma(-a1[o], b1[o], x1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) c0[sw(M::drow(lane, r), col)] = x0[r];
    if (two) {
#pragma unroll
        for (int r = 0; r < 4; ++r) c1[sw(M::drow(lane, r), col)] = x1[r];
    }
}

// Blocked right-looking factorisation of the LDS block triangle with
// lookahead: while waves 1..3 apply the trailing update of block column
// J, wave 0 first updates the next diagonal block and factors it, so the
// serial 16x16 factorisations overlap the MFMA work.  Two barriers per
// block column.  On return the diagonal slots hold D_J = L_JJ^{-1} and the
// off-diagonal slots L_IJ; each L_JJ goes to Lout when Lout != nullptr.
// Returns 0 or the 1-based failing row (LAPACK info).
template <typename T>
__device__ __forceinline__ int factor_blocked(T *L, int nb, int n, T *Lout, int64_t ldo, int *s_flag) {
    using M = Mfma16<T>;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto blk = [&](int I, int J) { return L + (tri(I) + J) * 256; };
    auto lout = [&](int J) { return (Lout != nullptr) ? Lout + 16 * J + (int64_t)16 * J * ldo : (T *)nullptr; };
    if (wave == 0) {
        const int f = factor_diag_block(blk(0, 0), lout(0), ldo, n);
        if (lane == 0) *s_flag = (f >= 0) ? f + 1 : 0;
    }
    __syncthreads();
    if (*s_flag) return *s_flag;
    for (int J = 0; J < nb; ++J) {
        const T *dJ = blk(J, J);
        // panel: L_IJ = A_IJ * D_J^T
        for (int I = J + 1 + wave; I < nb; I += kWaves) {
            T *t = blk(I, J);
            typename M::acc_t acc = M::zero();
            const int col = lane & 15;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int o = sw(col, (lane >> 4) + 4 * kk);
                acc = M::fma(t[o], dJ[o], acc);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) t[sw(M::drow(lane, r), col)] = acc[r];
        }
        __syncthreads();
        if (J + 1 == nb) break;
        if (wave == 0) {
            // lookahead: next diagonal tile first, then its factorisation
            tile_update2(blk(J + 1, J + 1), blk(J + 1, J), blk(J + 1, J), (T *)nullptr, (const T *)nullptr,
                         (const T *)nullptr, false);
            const int f = factor_diag_block(blk(J + 1, J + 1), lout(J + 1), ldo, n - 16 * (J + 1));
            if (lane == 0) *s_flag = (f >= 0) ? 16 * (J + 1) + f + 1 : 0;
        } else {
            // remaining tiles (I,K), J < K <= I, except (J+1,J+1), over waves 1..3
            int t = 0, pend = -1;
            T *pc = nullptr;
            const T *pa = nullptr, *pb = nullptr;
            for (int K = J + 1; K < nb; ++K) {
                for (int I = K; I < nb; ++I) {
                    if (I == J + 1 && K == J + 1) continue;
                    if ((t++ % (kWaves - 1)) != wave - 1) continue;
                    if (pend < 0) {
                        pc = blk(I, K);
                        pa = blk(I, J);
                        pb = blk(K, J);
                        pend = 1;
                    } else {
                        tile_update2(pc, pa, pb, blk(I, K), blk(I, J), blk(K, J), true);
                        pend = -1;
                    }
                }
            }
            if (pend > 0) tile_update2(pc, pa, pb, (T *)nullptr, (const T *)nullptr, (const T *)nullptr, false);
        }
        __syncthreads();
        if (*s_flag) return *s_flag;
    }
    return 0;
}

// In LDS, replace each diagonal block L_JJ by its inverse (wave J % 4).
template <typename T>
__device__ __forceinline__ void invert_diag_blocks(T *L, int nb) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int J = wave; J < nb; J += kWaves) {
        T *dJ = L + (tri(J) + J) * 256;
        T row[16], nx[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) row[c] = dJ[sw(lane & 15, c)];
        tri_inverse_steps<0>(row, T(1) / dJ[sw(lane & 15, lane & 15)], nx);
        if (lane < 16) {
#pragma unroll
            for (int r = 0; r < 16; ++r) dJ[sw(r, lane)] = -nx[r];
        }
    }
}

// y_i = sum_k M(i, k) v[k], or sum_k M(k, i) v[k] when TRANS (M = a D or L
// block), two partial sums.
template <bool TRANS, typename T>
__device__ __forceinline__ T dot16(const T *m, int i, const T *v) {
    T a0 = T(0), a1 = T(0);
#pragma unroll
    for (int k = 0; k < 16; k += 2) {
        a0 += m[TRANS ? sw(k, i) : sw(i, k)] * v[k];
        a1 += m[TRANS ? sw(k + 1, i) : sw(i, k + 1)] * v[k + 1];
    }
    return a0 + a1;
}

// Solve L L^T Y = Y in place for the npad x 4 block Y (LDS, column-major,
// ld = npad) with the block triangle (diagonal slots = inverses).  Lane =
// row + 16 * rhs inside a 16-row block.  Lookahead: the wave that owns the
// next block row applies the current update to it first and then its
// diagonal product, so each block step costs one barrier.
template <typename T>
__device__ __forceinline__ void solve_blocked(const T *L, int nb, T *Y) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, r = lane >> 4;
    const int ld = 16 * nb;
    auto blk = [&](int I, int J) { return L + (tri(I) + J) * 256; };
    // forward: L y = b
    if (wave == 0) {
        T *y = Y + ld * r;
        const T v = dot16<false>(blk(0, 0), i, y);
        y[i] = v;
    }
    __syncthreads();
    for (int I = 0; I + 1 < nb; ++I) {
        const T *yI = Y + 16 * I + ld * r;
        const int owner = (I + 1) & (kWaves - 1);
        if (wave == owner) {
            T *x = Y + 16 * (I + 1) + ld * r;
            x[i] -= dot16<false>(blk(I + 1, I), i, yI);
            const T v = dot16<false>(blk(I + 1, I + 1), i, x);
            x[i] = v;
        } else {
            int t = 0;
            for (int K = I + 2; K < nb; ++K, ++t) {
                if ((t % (kWaves - 1)) != ((wave - owner - 1) & (kWaves - 1))) continue;
                T *x = Y + 16 * K + ld * r;
                x[i] -= dot16<false>(blk(K, I), i, yI);
            }
        }
        __syncthreads();
    }
    // backward: L^T x = y
    const int last = nb - 1;
    if (wave == (last & (kWaves - 1))) {
        T *y = Y + 16 * last + ld * r;
        const T v = dot16<true>(blk(last, last), i, y);
        y[i] = v;
    }
    __syncthreads();
    for (int I = last; I > 0; --I) {
        const T *zI = Y + 16 * I + ld * r;
        const int owner = (I - 1) & (kWaves - 1);
        if (wave == owner) {
            T *x = Y + 16 * (I - 1) + ld * r;
            x[i] -= dot16<true>(blk(I, I - 1), i, zI);
            const T v = dot16<true>(blk(I - 1, I - 1), i, x);
            x[i] = v;
        } else {
            int t = 0;
            for (int K = I - 2; K >= 0; --K, ++t) {
                if ((t % (kWaves - 1)) != ((wave - owner - 1) & (kWaves - 1))) continue;
                T *x = Y + 16 * K + ld * r;
                x[i] -= dot16<true>(blk(I, K), i, zI);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ kernels --
// Factor only (API: CholeskyBatchFactoriser::factorise).
// n <= 64 leaves the LDS for many workgroups: four wavefronts per SIMD are
// worth a few spilled registers (4096 FP64 systems of n = 40: 118 us with
// two, 77 us with four).
template <typename T, int NB>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(NB <= 4 ? 4 : 2))) void potrf_kernel(int n, T *A, int64_t lda, int64_t strideA,
                                                         int *info, int64_t batch) {
    __shared__ T L[tri(NB) * 256];
    __shared__ int s_flag;
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    const int nb = (n + 15) >> 4;
    T *a = A + b * strideA;
    load_lower(a, lda, n, nb, L);
    __syncthreads();
    const int fail = factor_blocked(L, nb, n, a, lda, &s_flag);
    if (fail == 0) store_offdiag(a, lda, n, nb, L);
    if (threadIdx.x == 0 && info != nullptr) info[b] = fail;
}

// Solve only (API: CholeskyBatchFactoriser::solve), any nrhs.
template <typename T, int NB>
__global__ __launch_bounds__(kThreads) void potrs_kernel(int n, int nrhs, const T *Lg, int64_t lda,
                                                         int64_t strideL, T *B, int64_t ldb,
                                                         int64_t strideB, int *info, int64_t batch) {
    __shared__ T L[tri(NB) * 256];
    __shared__ T Y[16 * NB * kRhsChunk];
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    const int nb = (n + 15) >> 4;
    const int npad = 16 * nb;
    load_lower(Lg + b * strideL, lda, n, nb, L);
    __syncthreads();
    invert_diag_blocks(L, nb);
    T *bb = B + b * strideB;
    for (int r0 = 0; r0 < nrhs; r0 += kRhsChunk) {
        __syncthreads();
        for (int e = threadIdx.x; e < npad * kRhsChunk; e += kThreads) {
            const int row = e % npad, c = e / npad;
            Y[e] = (row < n && r0 + c < nrhs) ? bb[row + (int64_t)(r0 + c) * ldb] : T(0);
        }
        __syncthreads();
        solve_blocked(L, nb, Y);
        for (int e = threadIdx.x; e < npad * kRhsChunk; e += kThreads) {
            const int row = e % npad, c = e / npad;
            if (row < n && r0 + c < nrhs) bb[row + (int64_t)(r0 + c) * ldb] = Y[e];
        }
    }
    if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
}

// Fused factor + solve.  WRITE_L: A <- L (API shape).  X may alias B.
// mask != nullptr: only matrices with mask[b] < 0 are processed (the FP64
// fallback of the mixed solver); then A is read only.
template <typename T, int NB, bool WRITE_L>
__global__ __launch_bounds__(kThreads) void posv_kernel(int n, int nrhs, T *A, int64_t lda,
                                                        int64_t strideA, const T *B, int64_t ldb,
                                                        int64_t strideB, T *X, int64_t ldx,
                                                        int64_t strideX, int *info, int64_t batch,
                                                        const int *mask) {
    __shared__ T L[tri(NB) * 256];
    __shared__ T Y[16 * NB * kRhsChunk];
    __shared__ int s_flag;
    if (mask != nullptr) {
        // a masked launch mostly finds nothing to do: read this workgroup's
        // share of the mask at once (one entry per thread) instead of one
        // dependent load per matrix, and leave if none is selected
        const int64_t bt = blockIdx.x + (int64_t)threadIdx.x * gridDim.x;
        const int need = (bt < batch && mask[bt] < 0) ? 1 : 0;
        const bool covered = (int64_t)kThreads * gridDim.x >= batch;  // uniform
        if (!__syncthreads_or(need) && covered) return;
    }
    for (int64_t b = blockIdx.x; b < batch; b += gridDim.x) {
        if (mask != nullptr && mask[b] >= 0) continue;
        const int nb = (n + 15) >> 4;
        const int npad = 16 * nb;
        T *a = A + b * strideA;
        __syncthreads();
        load_lower(a, lda, n, nb, L);
        __syncthreads();
        const int fail = factor_blocked(L, nb, n, WRITE_L ? a : (T *)nullptr, lda, &s_flag);
        if (threadIdx.x == 0 && info != nullptr) info[b] = fail;
        if (fail) continue;  // uniform
        if (WRITE_L) store_offdiag(a, lda, n, nb, L);
        const T *bb = B + b * strideB;
        T *xx = X + b * strideX;
        for (int r0 = 0; r0 < nrhs; r0 += kRhsChunk) {
            __syncthreads();
            for (int e = threadIdx.x; e < npad * kRhsChunk; e += kThreads) {
                const int row = e % npad, c = e / npad;
                Y[e] = (row < n && r0 + c < nrhs) ? bb[row + (int64_t)(r0 + c) * ldb] : T(0);
            }
            __syncthreads();
            solve_blocked(L, nb, Y);
            for (int e = threadIdx.x; e < npad * kRhsChunk; e += kThreads) {
                const int row = e % npad, c = e / npad;
                if (row < n && r0 + c < nrhs) xx[row + (int64_t)(r0 + c) * ldx] = Y[e];
            }
        }
    }
}

// ------------------------------------------------- larger n, one workgroup --
// n in (128, kStripMaxN]: the block triangle no longer fits the LDS, so L
// stays in global memory (one matrix is a few hundred KB: L2 resident) and
// the factorisation is left-looking by block columns of 16.  Eight
// wavefronts: wave 0 factors the diagonal blocks, the others own the
// 16-row strips I = (wave - 1) + 7 s.  What bounds it is the chain of
// diagonal blocks (16 dependent pivots each), so everything else runs
// beside it: while wave 0 factors block J, the strips finish column J with
// the block product of column J - 1 and form column J + 1 up to K = J - 1
// from L in global memory.  Two barriers per block column, no trailing
// matrix is written back.  A strip's column is kept transposed (lane % 16 =
// row, items = columns): that is the accumulator layout of
// D[j][i] = sum_k L_J[j][k] L_I[i][k], it is a B operand for the next
// product without any data movement, and its loads and stores are
// contiguous down a column.
// 256 systems of n = 200 in FP64, factorisation: the unblocked kernel that
// read and wrote the whole trailing matrix for each column took 3424 us,
// this one 70 us.
constexpr int kStripThreads = 512;
constexpr int kStripWorkers = kStripThreads / kWave - 1;
constexpr int kStripSlots = 6;  // strips per wavefront; FP64 has 31 registers in scratch here already
constexpr int64_t kStripMaxN = 16 * kStripWorkers * kStripSlots;
static_assert(kStripMaxN <= 2 * kStripThreads, "potrs_strips_kernel holds two rows a thread");
constexpr int64_t kStripMaxLd = 1 << 26;  // lane offsets of up to 13 columns are 32-bit

// Two strips in FP64 fit the registers of two workgroups per CU.
template <typename T, int S>
__global__ __launch_bounds__(kStripThreads) __attribute__((amdgpu_waves_per_eu(S == 2 ? 4 : 2))) void potrf_strips_kernel(int n, T *A, int64_t lda, int64_t strideA,
                                                                     int *info, int64_t batch) {
    using M = Mfma16<T>;
    __shared__ T dg[2][256];  // diagonal block J, then its inverse (slot J & 1)
    __shared__ T lo[256];     // L_{J+1,J}
    __shared__ int s_flag;
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    T *a = A + b * strideA;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wave - 1;
    const int c = lane & 15;
    const int nb = (n + 15) >> 4;
    if (threadIdx.x < 256) {
        const int i = threadIdx.x & 15, k = threadIdx.x >> 4;
        dg[0][sw(i, k)] = (i >= k) ? a[i + (int64_t)k * lda] : T(0);  // n > 16
    }
    if (wave == 0) {
        // the diagonal chain; its barriers pair with the workers' below
        __syncthreads();
        int fail = 0;
#pragma unroll 1
        for (int J = 0; J < nb; ++J) {
            const int f = factor_diag_block<true>(dg[J & 1], a + 16 * J + (int64_t)16 * J * lda, lda, n - 16 * J);
            fail = (f >= 0) ? 16 * J + f + 1 : 0;  // uniform
            if (lane == 0) s_flag = fail;
            __syncthreads();
            if (fail != 0 || J + 1 == nb) break;
            __syncthreads();
        }
        if (lane == 0 && info != nullptr) info[b] = fail;
        return;
    }
    typename M::acc_t acc[S], nxt[S], lr[S];  // column J, column J + 1 so far, L_{I,J-1}
    // Step t of a 16x16 block takes column drow(lane, t) = drow(lane, 0) +
    // drow(0, t) of it: uniform column pointers plus one 32-bit lane offset
    // per strip (its row, clamped into the matrix: what a lane past n
    // computes stays in its own row and is not stored).
    unsigned rs[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        acc[s] = nxt[s] = lr[s] = M::zero();
        const int r = 16 * (w + kStripWorkers * s) + c;
        rs[s] = (unsigned)((r < n ? r : n - 1) + M::drow(lane, 0) * (int)lda);
    }
    // A_{I,J}: slots past their strips' turn load and compute too, so that
    // no branch splits the accumulators; nothing of theirs is used.  Entries
    // above the diagonal of A_{J,J} stay above it.  The last block column
    // (only its diagonal block is left) must not be read past column n.
    auto load_block = [&](int s, int J) {
        typename M::acc_t v;
        const T *p = a + (int64_t)16 * J * lda;
        if (J + 1 < nb) {
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = (p + M::drow(0, t) * lda)[rs[s]];
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                v[t] = (16 * J + M::drow(lane, t) < n) ? (p + M::drow(0, t) * lda)[rs[s]] : T(0);
        }
        return v;
    };
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = load_block(s, 0);
    __syncthreads();
#pragma unroll 1
    for (int J = 0; J < nb; ++J) {
        if (J > 0) {
            T lj[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) lj[t] = -lo[sw(c, M::drow(lane, t))];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int s = 0; s < S; ++s) acc[s] = M::fma(lj[t], lr[s][t], acc[s]);
        }
        if (J + 1 < nb) {
            // column J + 1 over K < J
#pragma unroll
            for (int s = 0; s < S; ++s) nxt[s] = load_block(s, J + 1);
            const int rj = 16 * (J + 1) + c;
            const unsigned pj = (unsigned)((rj < n ? rj : n - 1) + M::drow(lane, 0) * (int)lda);
            // the strips still below column J + 1 are the slots from
            // `first` on: one loop for each, without branches inside
            auto sum_columns = [&](auto first_c) {
                constexpr int first = decltype(first_c)::value;
                const T *ak = a;
#pragma unroll 1
                for (int K = 0; K < J; ++K, ak += 16 * lda) {
                    T x[4], y[S][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) x[t] = -(ak + M::drow(0, t) * lda)[pj];
#pragma unroll
                    for (int s = first; s < S; ++s)
#pragma unroll
                        for (int t = 0; t < 4; ++t) y[s][t] = (ak + M::drow(0, t) * lda)[rs[s]];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int s = first; s < S; ++s) nxt[s] = M::fma(x[t], y[s][t], nxt[s]);
                }
            };
            const int first = (J - w) < 0 ? 0 : (J - w) / kStripWorkers + 1;  // S or more: none left here
            if (first == 0) sum_columns(std::integral_constant<int, 0>());
            else if (first == 1) sum_columns(std::integral_constant<int, 1>());
            if constexpr (S > 2) {
                if (first == 2) sum_columns(std::integral_constant<int, 2>());
                else if (first == 3) sum_columns(std::integral_constant<int, 3>());
            }
            if constexpr (S > 4) {
                if (first == 4) sum_columns(std::integral_constant<int, 4>());
                else if (first == 5) sum_columns(std::integral_constant<int, 5>());
            }
        }
        __syncthreads();
        if (s_flag != 0 || J + 1 == nb) break;  // uniform
        const T *D = dg[J & 1];
        T d[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) d[t] = D[sw(c, M::drow(lane, t))];
        T *pl = a + (int64_t)16 * J * lda;
#pragma unroll
        for (int s = 0; s < S; ++s) lr[s] = M::zero();
        // L_IJ^T = D_J (A_IJ - ...)^T
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int s = 0; s < S; ++s) lr[s] = M::fma(d[t], acc[s][t], lr[s]);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int I = w + kStripWorkers * s;
            if (I == J + 1) {
                typename M::acc_t q = nxt[s];
#pragma unroll
                for (int t = 0; t < 4; ++t) q = M::fma(-lr[s][t], lr[s][t], q);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int j = M::drow(lane, t), gi = 16 * I + c, gk = 16 * I + j;
                    lo[sw(c, j)] = lr[s][t];
                    dg[(J + 1) & 1][sw(c, j)] = (gi < n && gk < n) ? q[t] : ((c == j) ? T(1) : T(0));
                }
            }
            if (I > J && 16 * I + c < n) {
#pragma unroll
                for (int t = 0; t < 4; ++t) (pl + M::drow(0, t) * lda)[rs[s]] = lr[s][t];
            }
            acc[s] = nxt[s];
        }
        __syncthreads();
    }
}

// L L^T x = b by columns for each right-hand side, one workgroup of NT threads;
// red: NT elements of LDS.
template <int NT, typename T>
__device__ __forceinline__ void substitute(int n, int nrhs, const T *l, int64_t lda, T *B, int64_t ldb, T *red) {
    for (int r = 0; r < nrhs; ++r) {
        T *x = B + (int64_t)r * ldb;
        for (int k = 0; k < n; ++k) {
            __syncthreads();
            const T xk = x[k] / l[k + (int64_t)k * lda];
            __syncthreads();
            if (threadIdx.x == 0) x[k] = xk;
            for (int i = k + 1 + threadIdx.x; i < n; i += NT) x[i] -= l[i + (int64_t)k * lda] * xk;
        }
        for (int k = n - 1; k >= 0; --k) {
            __syncthreads();
            // x_k = (x_k - sum_{i>k} l_ik x_i) / l_kk : block reduction
            T part = T(0);
            for (int i = k + 1 + threadIdx.x; i < n; i += NT) part += l[i + (int64_t)k * lda] * x[i];
            red[threadIdx.x] = part;
            __syncthreads();
            for (int s = NT / 2; s > 0; s >>= 1) {
                if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
                __syncthreads();
            }
            if (threadIdx.x == 0) x[k] = (x[k] - red[0]) / l[k + (int64_t)k * lda];
        }
    }
}

// Solve with the factor of a larger matrix (n in (128, kStripMaxN]) for any
// nrhs, four right-hand sides per pass.  The reference substitution is a
// chain of 2 n dependent steps; here the diagonal blocks are inverted first
// (all at once, one wavefront each), so a pass is a chain of 2 n / 16
// block steps.  Forward: the thread that owns row i keeps its four values
// in registers and subtracts block column J (its 16 entries of L loaded a
// step ahead); the wavefront that owns the next block row then multiplies
// it by its inverse, one barrier per step.  Backward: wavefront w forms the
// dot products of columns 2 w and 2 w + 1 of block J with the solution below
// (rows along the lanes, so L is read contiguously), two barriers per step.
// 256 systems of n = 200 in FP64, one right-hand side: 310 us for the
// substitution by columns with two barriers and a tree reduction each,
// 49 us now.
// skip != nullptr: systems with skip[b] != 0 (a failed factorisation) are
// left as they are, as LAPACK dposv leaves B.
// A factor with a diagonal entry that has no normal reciprocal is substituted
// by columns, with divisions.
// ROWS: rows of a thread, n <= ROWS * kStripThreads.
template <typename T, int ROWS>
__global__ __launch_bounds__(kStripThreads) void potrs_strips_kernel(int n, int nrhs, const T *L, int64_t lda,
                                                                     int64_t strideL, T *B, int64_t ldb,
                                                                     int64_t strideB, int *info, int64_t batch,
                                                                     const int *skip) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_strips[];
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    if (skip != nullptr && skip[b] != 0) return;
    constexpr int kStripWaves = kStripThreads / kWave;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int nb = (n + 15) >> 4, npad = 16 * nb;
    T *D = reinterpret_cast<T *>(dyn_strips);  // nb inverses of 16x16 (sw order)
    T *Y = D + 256 * nb;                       // npad x 4
    T *Z = Y + npad * kRhsChunk;               // 16 x 4 sums of the backward step
    const T *l = L + b * strideL;
    bool divide = false;
    for (int J = wave; J < nb; J += kStripWaves) {
        T row[16], nx[16];
        const int gi = 16 * J + c;
#pragma unroll
        for (int k = 0; k < 16; ++k)
            row[k] = (gi < n && c >= k) ? l[gi + (int64_t)(16 * J + k) * lda] : ((c == k) ? T(1) : T(0));
        const T d = (gi < n) ? l[gi + (int64_t)gi * lda] : T(1);
        divide = divide || !hh::has_reciprocal(d);
        tri_inverse_steps<0>(row, T(1) / d, nx);
        if (lane < 16) {
#pragma unroll
            for (int r = 0; r < 16; ++r) D[256 * J + sw(r, lane)] = -nx[r];
        }
    }
    T *bb = B + b * strideB;
    int *flag = reinterpret_cast<int *>(Z);  // one for each wavefront
    divide = __any(divide);
    if (lane == 0) flag[wave] = divide;
    __syncthreads();
    if (__builtin_expect(__any(lane < kStripWaves && flag[lane]), 0)) {  // the same in every wavefront
        __syncthreads();
        substitute<kStripThreads>(n, nrhs, l, lda, bb, ldb, D);  // 256 nb > kStripThreads
        if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
        return;
    }
    for (int r0 = 0; r0 < nrhs; r0 += kRhsChunk) {
        if (r0 > 0) __syncthreads();
        for (int e = threadIdx.x; e < npad * kRhsChunk; e += kStripThreads) {
            const int row = e % npad, col = e / npad;
            Y[e] = (row < n && r0 + col < nrhs) ? bb[row + (int64_t)(r0 + col) * ldb] : T(0);
        }
        __syncthreads();
        // forward: this thread's rows and their entries of block column 0
        T x[ROWS][kRhsChunk], lc[ROWS][16];
        auto load_col = [&](int J) {
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                const int i = threadIdx.x + kStripThreads * u;
                if (i >= 16 * (J + 1) && i < n) {
#pragma unroll
                    for (int k = 0; k < 16; ++k) lc[u][k] = l[i + (int64_t)(16 * J + k) * lda];
                }
            }
        };
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            const int i = threadIdx.x + kStripThreads * u;
#pragma unroll
            for (int r = 0; r < kRhsChunk; ++r) x[u][r] = (i < n) ? Y[i + npad * r] : T(0);
        }
        load_col(0);
        if (wave == 0) {
            const T v = dot16<false>(D, c, Y + npad * g);
            Y[c + npad * g] = v;
        }
        __syncthreads();
        for (int J = 0; J + 1 < nb; ++J) {
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                const int i = threadIdx.x + kStripThreads * u;
                if (i >= 16 * (J + 1) && i < n) {
#pragma unroll
                    for (int r = 0; r < kRhsChunk; ++r) {
                        const T *y = Y + 16 * J + npad * r;
                        T s0 = T(0), s1 = T(0);
#pragma unroll
                        for (int k = 0; k < 16; k += 2) {
                            s0 += lc[u][k] * y[k];
                            s1 += lc[u][k + 1] * y[k + 1];
                        }
                        x[u][r] -= s0 + s1;
                    }
                    // the next block row goes through its inverse below
                    if (i < 16 * (J + 2)) {
#pragma unroll
                        for (int r = 0; r < kRhsChunk; ++r) Y[i + npad * r] = x[u][r];
                    }
                }
            }
            if (J + 2 < nb) load_col(J + 1);
            if (wave == (((J + 1) >> 2) & (kStripWaves - 1))) {  // holds rows 16 (J + 1) ..
                hh::wave_sync();
                T *y = Y + 16 * (J + 1) + npad * g;
                const T v = dot16<false>(D + 256 * (J + 1), c, y);
                hh::wave_sync();
                y[c] = v;
            }
            __syncthreads();
        }
        // backward
        for (int J = nb - 1; J >= 0; --J) {
            if (J + 1 < nb) {
                T s[2][kRhsChunk];
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int r = 0; r < kRhsChunk; ++r) s[q][r] = T(0);
                for (int i = 16 * (J + 1) + lane; i < n; i += kWave) {
                    T lv[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) lv[q] = l[i + (int64_t)(16 * J + 2 * wave + q) * lda];
#pragma unroll
                    for (int r = 0; r < kRhsChunk; ++r) {
                        const T y = Y[i + npad * r];
#pragma unroll
                        for (int q = 0; q < 2; ++q) s[q][r] += lv[q] * y;
                    }
                }
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int r = 0; r < kRhsChunk; ++r) s[q][r] = wave_sum(s[q][r]);
                if (lane == 0) {
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int r = 0; r < kRhsChunk; ++r) Z[2 * wave + q + 16 * r] = s[q][r];
                }
                __syncthreads();
            }
            if (wave == 0) {
                T *y = Y + 16 * J + npad * g;
                T v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = y[k] - ((J + 1 < nb) ? Z[k + 16 * g] : T(0));
                T s0 = T(0), s1 = T(0);
#pragma unroll
                for (int k = 0; k < 16; k += 2) {
                    s0 += D[256 * J + sw(k, c)] * v[k];
                    s1 += D[256 * J + sw(k + 1, c)] * v[k + 1];
                }
                hh::wave_sync();
                y[c] = s0 + s1;
            }
            __syncthreads();
        }
        for (int e = threadIdx.x; e < npad * kRhsChunk; e += kStripThreads) {
            const int row = e % npad, col = e / npad;
            if (row < n && r0 + col < nrhs) bb[row + (int64_t)(r0 + col) * ldb] = Y[e];
        }
    }
    if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
}

// ----------------------------------------------- large-n global kernels --
// Correctness path for what the strips do not take: unblocked right-looking algorithm on
// the matrix in global memory, one workgroup per matrix.
template <typename T>
__global__ __launch_bounds__(kThreads) void potrf_global_kernel(int n, T *A, int64_t lda,
                                                                int64_t strideA, int *info,
                                                                int64_t batch) {
    __shared__ int s_fail;
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    T *a = A + b * strideA;
    if (threadIdx.x == 0) s_fail = 0;
    for (int k = 0; k < n; ++k) {
        __syncthreads();
        const T d = a[k + (int64_t)k * lda];
        if (!(d > T(0))) {
            if (threadIdx.x == 0) s_fail = k + 1;
            break;
        }
        const T s = dev_sqrt(d);
        __syncthreads();
        for (int i = k + 1 + threadIdx.x; i < n; i += kThreads) a[i + (int64_t)k * lda] /= s;
        if (threadIdx.x == 0) a[k + (int64_t)k * lda] = s;
        __syncthreads();
        const int m = n - k - 1;
        for (int64_t e = threadIdx.x; e < (int64_t)m * m; e += kThreads) {
            const int i = k + 1 + (int)(e % m), j = k + 1 + (int)(e / m);
            if (i >= j) a[i + (int64_t)j * lda] -= a[i + (int64_t)k * lda] * a[j + (int64_t)k * lda];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && info != nullptr) info[b] = s_fail;
}

// skip as in potrs_strips_kernel.
template <typename T>
__global__ __launch_bounds__(kThreads) void potrs_global_kernel(int n, int nrhs, const T *L,
                                                                int64_t lda, int64_t strideL, T *B,
                                                                int64_t ldb, int64_t strideB,
                                                                int *info, int64_t batch,
                                                                const int *skip) {
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    if (skip != nullptr && skip[b] != 0) return;
    __shared__ T red[kThreads];
    substitute<kThreads>(n, nrhs, L + b * strideL, lda, B + b * strideB, ldb, red);
    if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
}

// Copies the rows x cols matrices src_b (ld lds) to dst_b (ld ldd).
template <typename T>
__global__ __launch_bounds__(kThreads) void copy_batch_kernel(int rows, int cols, const T *__restrict__ src,
                                                              int64_t lds, int64_t strideS, T *__restrict__ dst,
                                                              int64_t ldd, int64_t strideD, int64_t batch) {
    const int64_t per = (int64_t)rows * cols;
    for (int64_t b = blockIdx.x; b < batch; b += gridDim.x)
        for (int64_t e = threadIdx.x; e < per; e += kThreads) {
            const int64_t i = e % rows, j = e / rows;
            dst[b * strideD + i + j * ldd] = src[b * strideS + i + j * lds];
        }
}

// ----------------------------------------------------------- dispatch --
template <typename T>
int potrf_dispatch(int64_t n, T *A, int64_t lda, int64_t strideA, int *info, int64_t batch,
                   hipStream_t st) {
    // factor only: the register-resident small kernel with no right-hand
    // sides (B and X are not read or written when nrhs = 0)
    if (n <= 32)
        return chols::launch_posv_small<T>((int)n, 0, A, lda, strideA, A, lda, strideA, A, lda, strideA, info, batch,
                                           nullptr, true, st);
    // n > 32 from here on (smaller n returned above)
    const dim3 grid((unsigned)batch), block(kThreads);
    if (n <= 48) hipLaunchKernelGGL((potrf_kernel<T, 3>), grid, block, 0, st, (int)n, A, lda, strideA, info, batch);
    else if (n <= 64) hipLaunchKernelGGL((potrf_kernel<T, 4>), grid, block, 0, st, (int)n, A, lda, strideA, info, batch);
    else if (n <= 128) hipLaunchKernelGGL((potrf_kernel<T, 8>), grid, block, 0, st, (int)n, A, lda, strideA, info, batch);
    else if (lda > kStripMaxLd || n > kStripMaxN)
        hipLaunchKernelGGL((potrf_global_kernel<T>), grid, block, 0, st, (int)n, A, lda, strideA, info, batch);
    else if (n <= 16 * kStripWorkers * 2)
        hipLaunchKernelGGL((potrf_strips_kernel<T, 2>), grid, dim3(kStripThreads), 0, st, (int)n, A, lda, strideA, info, batch);
    else if (n <= 16 * kStripWorkers * 4)
        hipLaunchKernelGGL((potrf_strips_kernel<T, 4>), grid, dim3(kStripThreads), 0, st, (int)n, A, lda, strideA, info, batch);
    else
        hipLaunchKernelGGL((potrf_strips_kernel<T, kStripSlots>), grid, dim3(kStripThreads), 0, st, (int)n, A, lda, strideA, info, batch);
    return launch_check("potrf_kernel");
}

// The solve for n > 128; skip as in the kernels.
template <typename T>
int potrs_large(int64_t n, int64_t nrhs, const T *L, int64_t lda, int64_t strideL, T *B, int64_t ldb,
                int64_t strideB, int *info, int64_t batch, const int *skip, hipStream_t st) {
    const int64_t nb = ceil_div(n, 16);
    if (n <= kStripMaxN) {
        // at most 108 KB of LDS (n = kStripMaxN in FP64)
        auto bytes = [](int64_t blocks) {
            return sizeof(T) * (size_t)(256 * blocks + 16 * blocks * kRhsChunk + 16 * kRhsChunk);
        };
        const size_t lds = bytes(nb);
        auto kern = n <= kStripThreads ? potrs_strips_kernel<T, 1> : potrs_strips_kernel<T, 2>;
        // the same value from every call: another thread's launch of this kernel
        // may come between this line and the next
        if (lds > 64 * 1024)
            GPUTILS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes(kStripMaxN / 16)));
        hipLaunchKernelGGL(kern, dim3((unsigned)batch), dim3(kStripThreads), lds, st, (int)n, (int)nrhs, L, lda,
                           strideL, B, ldb, strideB, info, batch, skip);
        return launch_check("potrs_strips_kernel");
    }
    hipLaunchKernelGGL((potrs_global_kernel<T>), dim3((unsigned)batch), dim3(kThreads), 0, st, (int)n, (int)nrhs, L,
                       lda, strideL, B, ldb, strideB, info, batch, skip);
    return launch_check("potrs_global_kernel");
}

template <typename T>
int potrs_dispatch(int64_t n, int64_t nrhs, const T *L, int64_t lda, int64_t strideL, T *B,
                   int64_t ldb, int64_t strideB, int *info, int64_t batch, hipStream_t st) {
    if (n <= 32)
        return chols::launch_potrs_small<T>((int)n, (int)nrhs, L, lda, strideL, B, ldb, strideB, info, batch, st);
    const dim3 grid((unsigned)batch), block(kThreads);
#define GPUTILS_POTRS(NBV) \
    hipLaunchKernelGGL((potrs_kernel<T, NBV>), grid, block, 0, st, (int)n, (int)nrhs, L, lda, strideL, B, ldb, strideB, info, batch)
    // n > 32 from here on (smaller n returned above)
    if (n <= 48) GPUTILS_POTRS(3);
    else if (n <= 64) GPUTILS_POTRS(4);
    else if (n <= 128) GPUTILS_POTRS(8);
    else return potrs_large<T>(n, nrhs, L, lda, strideL, B, ldb, strideB, info, batch, nullptr, st);
#undef GPUTILS_POTRS
    return launch_check("potrs_kernel");
}

template <typename T, bool WRITE_L>
int posv_dispatch(int64_t n, int64_t nrhs, T *A, int64_t lda, int64_t strideA, const T *B,
                  int64_t ldb, int64_t strideB, T *X, int64_t ldx, int64_t strideX, int *info,
                  int64_t batch, const int *mask, hipStream_t st) {
    if (n <= 32)
        return chols::launch_posv_small<T>((int)n, (int)nrhs, A, lda, strideA, B, ldb, strideB, X, ldx, strideX, info,
                                           batch, mask, WRITE_L, st);
    // masked (fallback) launches scan the mask with a grid-stride loop: two
    // workgroups per CU fill the GPU at this kernel's LDS size
    const int64_t g = (mask != nullptr) ? (batch < 512 ? batch : 512) : batch;
    const dim3 grid((unsigned)g), block(kThreads);
#define GPUTILS_POSV(NBV)                                                                     \
    hipLaunchKernelGGL((posv_kernel<T, NBV, WRITE_L>), grid, block, 0, st, (int)n, (int)nrhs, A, \
                       lda, strideA, B, ldb, strideB, X, ldx, strideX, info, batch, mask)
    // n > 32 from here on (smaller n returned above); n <= 128 (checked by
    // the callers)
    if (n <= 48) GPUTILS_POSV(3);
    else if (n <= 64) GPUTILS_POSV(4);
    else GPUTILS_POSV(8);
#undef GPUTILS_POSV
    return launch_check("posv_kernel");
}

}  // namespace chol
}  // namespace gputils

using namespace gputils;

extern "C" {

int gputils_spotrf_batched(int64_t n, float *A, int64_t lda, int64_t strideA, int *info,
                           int64_t batch, void *stream) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 3, "lda < max(1,n)");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, 6, "batch out of range");
    if (n == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(A != nullptr, 2, "A is NULL");
    return chol::potrf_dispatch<float>(n, A, lda, strideA, info, batch, as_stream(stream));
}

int gputils_dpotrf_batched(int64_t n, double *A, int64_t lda, int64_t strideA, int *info,
                           int64_t batch, void *stream) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 3, "lda < max(1,n)");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, 6, "batch out of range");
    if (n == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(A != nullptr, 2, "A is NULL");
    return chol::potrf_dispatch<double>(n, A, lda, strideA, info, batch, as_stream(stream));
}

int gputils_spotrs_batched(int64_t n, int64_t nrhs, const float *L, int64_t lda, int64_t strideL,
                           float *B, int64_t ldb, int64_t strideB, int *info, int64_t batch,
                           void *stream) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(nrhs >= 0, 2, "nrhs < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 4, "lda < max(1,n)");
    GPUTILS_ARG(ldb >= (n > 1 ? n : 1), 7, "ldb < max(1,n)");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, 10, "batch out of range");
    if (n == 0 || nrhs == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(L != nullptr, 3, "L is NULL");
    GPUTILS_ARG(B != nullptr, 6, "B is NULL");
    return chol::potrs_dispatch<float>(n, nrhs, L, lda, strideL, B, ldb, strideB, info, batch,
                                       as_stream(stream));
}

int gputils_dpotrs_batched(int64_t n, int64_t nrhs, const double *L, int64_t lda, int64_t strideL,
                           double *B, int64_t ldb, int64_t strideB, int *info, int64_t batch,
                           void *stream) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(nrhs >= 0, 2, "nrhs < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 4, "lda < max(1,n)");
    GPUTILS_ARG(ldb >= (n > 1 ? n : 1), 7, "ldb < max(1,n)");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, 10, "batch out of range");
    if (n == 0 || nrhs == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(L != nullptr, 3, "L is NULL");
    GPUTILS_ARG(B != nullptr, 6, "B is NULL");
    return chol::potrs_dispatch<double>(n, nrhs, L, lda, strideL, B, ldb, strideB, info, batch,
                                        as_stream(stream));
}

int gputils_dposv_batched(int64_t n, int64_t nrhs, double *A, int64_t lda, int64_t strideA,
                          double *B, int64_t ldb, int64_t strideB, int *info, int64_t batch,
                          void *stream) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(nrhs >= 0, 2, "nrhs < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 4, "lda < max(1,n)");
    GPUTILS_ARG(ldb >= (n > 1 ? n : 1), 7, "ldb < max(1,n)");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, 10, "batch out of range");
    if (n == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(A != nullptr, 3, "A is NULL");
    GPUTILS_ARG(nrhs == 0 || B != nullptr, 6, "B is NULL");
    hipStream_t st = as_stream(stream);
    if (n > 128) {
        // global-memory factor, then the solve of the systems it factorised
        // (a failed one keeps its B); info holds the factor's status
        GPUTILS_ARG(info != nullptr, 9, "info is NULL (needed for n > 128)");
        const int rc = chol::potrf_dispatch<double>(n, A, lda, strideA, info, batch, st);
        if (rc != GPUTILS_OK || nrhs == 0) return rc;
        return chol::potrs_large<double>(n, nrhs, A, lda, strideA, B, ldb, strideB, nullptr, batch, info, st);
    }
    return chol::posv_dispatch<double, true>(n, nrhs, A, lda, strideA, B, ldb, strideB, B, ldb,
                                             strideB, info, batch, nullptr, st);
}

int64_t gputils_dposv_mixed_workspace_bytes(int64_t n, int64_t batch) {
    if (n < 0 || batch < 0) return -1;
    return n <= cholw::kMixedMaxN ? 0 : n * n * (int64_t)sizeof(double) * batch;
}

}  // extern "C"

namespace {

// Arguments of the mixed solve after their checks; work is the FP64 copy
// of A for n > kMixedMaxN (the only device memory besides the caller's).
int posv_mixed_run(int64_t n, int64_t nrhs, const double *A, int64_t lda, int64_t strideA, const double *B,
                   int64_t ldb, int64_t strideB, double *X, int64_t ldx, int64_t strideX, double tol, int max_iter,
                   int *iters, int *info, double *work, int64_t batch, void *stream) {
    hipStream_t st = as_stream(stream);
    if (n > cholw::kMixedMaxN) {
        // beyond the fused kernel: FP64 factor and solve of copies (A and B
        // stay read only), every system reported as solved by the fallback
        double *L = work;
        const unsigned blocks = (unsigned)(batch < 4096 ? batch : 4096);
        hipLaunchKernelGGL((chol::copy_batch_kernel<double>), dim3(blocks), dim3(chol::kThreads), 0, st, (int)n, (int)n, A,
                           lda, strideA, L, n, n * n, batch);
        hipLaunchKernelGGL((chol::copy_batch_kernel<double>), dim3(blocks), dim3(chol::kThreads), 0, st, (int)n, (int)nrhs,
                           B, ldb, strideB, X, ldx, strideX, batch);
        int rc = launch_check("copy_batch_kernel");
        if (rc != GPUTILS_OK) return rc;
        rc = gputils_fill_bytes_async(iters, 0xff, (size_t)batch * sizeof(int), stream);  // iters = -1
        if (rc != GPUTILS_OK) return rc;
        rc = chol::potrf_dispatch<double>(n, L, n, n * n, info, batch, st);
        if (rc != GPUTILS_OK) return rc;
        return chol::potrs_dispatch<double>(n, nrhs, L, n, n * n, X, ldx, strideX, nullptr, batch, st);
    }
    int rc = cholw::launch_posv_mixed((int)n, (int)nrhs, A, lda, strideA, B, ldb, strideB, X, ldx, strideX, tol,
                                      max_iter, iters, info, batch, st);
    if (rc != GPUTILS_OK) return rc;
    // FP64 fallback for matrices flagged with iters < 0 (A, B read only)
    return chol::posv_dispatch<double, false>(n, nrhs, const_cast<double *>(A), lda, strideA, B, ldb,
                                              strideB, X, ldx, strideX, info, batch, iters, st);
}

// The argument checks both mixed entry points share (their argument
// numbers agree up to info, 15).
int posv_mixed_check(int64_t n, int64_t nrhs, const double *A, int64_t lda, const double *B, int64_t ldb,
                     const double *X, int64_t ldx, double tol, int max_iter, const int *iters, const int *info,
                     int64_t batch, int batch_arg) {
    GPUTILS_ARG(n >= 0, 1, "n < 0");
    GPUTILS_ARG(nrhs >= 0, 2, "nrhs < 0");
    GPUTILS_ARG(lda >= (n > 1 ? n : 1), 4, "lda < max(1,n)");
    GPUTILS_ARG(ldb >= (n > 1 ? n : 1), 7, "ldb < max(1,n)");
    GPUTILS_ARG(ldx >= (n > 1 ? n : 1), 10, "ldx < max(1,n)");
    GPUTILS_ARG(tol > 0.0, 12, "tol <= 0");
    GPUTILS_ARG(max_iter >= 0, 13, "max_iter < 0");
    GPUTILS_ARG(batch >= 0 && batch <= 0x7fffffff, batch_arg, "batch out of range");
    if (n == 0 || nrhs == 0 || batch == 0) return GPUTILS_OK;
    GPUTILS_ARG(A != nullptr, 3, "A is NULL");
    GPUTILS_ARG(B != nullptr, 6, "B is NULL");
    GPUTILS_ARG(X != nullptr, 9, "X is NULL");
    GPUTILS_ARG(iters != nullptr, 14, "iters is NULL");
    GPUTILS_ARG(info != nullptr, 15, "info is NULL");
    return GPUTILS_OK;
}

// Scratch of gputils_dposv_mixed_batched_noalloc: the FP64 copies of A that
// systems beyond the fused kernel (n > kMixedMaxN) are factorised in.  Each
// GPU holds its own copy for the life of the process; every call on one GPU
// uses the same array.
constexpr int64_t kNoallocScratchBytes = 16ll << 20;
static __device__ __align__(256) double scratch[kNoallocScratchBytes / sizeof(double)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
double *g_scratch_addr[kMaxDevices] = {};  // device address of `scratch`, per device

// The device address of `scratch` on the current device, looked up once per
// device (the host name of the array is only a stand-in for it).
int scratch_on_current_device(double **addr) {
    int dev = -1;
    GPUTILS_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("device %d is beyond the %d devices the allocation-free entry point supports", dev, kMaxDevices);
        return 1;
    }
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (g_scratch_addr[dev] == nullptr) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_error("hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return e != hipSuccess ? (int)e : 1;
        }
        g_scratch_addr[dev] = static_cast<double *>(p);
    }
    *addr = g_scratch_addr[dev];
    return GPUTILS_OK;
}

}  // namespace

extern "C" {

int gputils_dposv_mixed_batched(int64_t n, int64_t nrhs, const double *A, int64_t lda,
                                int64_t strideA, const double *B, int64_t ldb, int64_t strideB,
                                double *X, int64_t ldx, int64_t strideX, double tol, int max_iter,
                                int *iters, int *info, void *work, int64_t batch, void *stream) {
    int rc = posv_mixed_check(n, nrhs, A, lda, B, ldb, X, ldx, tol, max_iter, iters, info, batch, 17);
    if (rc != GPUTILS_OK || n == 0 || nrhs == 0 || batch == 0) return rc;
    GPUTILS_ARG(n <= cholw::kMixedMaxN || work != nullptr, 16,
                "work is NULL (query gputils_dposv_mixed_workspace_bytes)");
    return posv_mixed_run(n, nrhs, A, lda, strideA, B, ldb, strideB, X, ldx, strideX, tol, max_iter, iters, info,
                          static_cast<double *>(work), batch, stream);
}

int gputils_dposv_mixed_batched_noalloc(int64_t n, int64_t nrhs, const double *A, int64_t lda, int64_t strideA,
                                        const double *B, int64_t ldb, int64_t strideB, double *X, int64_t ldx,
                                        int64_t strideX, double tol, int max_iter, int *iters, int *info,
                                        int64_t batch, void *stream) {
    int rc = posv_mixed_check(n, nrhs, A, lda, B, ldb, X, ldx, tol, max_iter, iters, info, batch, 16);
    if (rc != GPUTILS_OK || n == 0 || nrhs == 0 || batch == 0) return rc;
    double *work = nullptr;
    if (n > cholw::kMixedMaxN) {
        // n <= 1448 keeps n*n*8*batch inside int64 for any batch <= 2^31
        GPUTILS_ARG(n <= 1448 && n * n * (int64_t)sizeof(double) * batch <= kNoallocScratchBytes, 16,
                    "n*n*batch*8 bytes exceed the 16 MiB scratch of gputils_dposv_mixed_batched_noalloc");
        rc = scratch_on_current_device(&work);
        if (rc != GPUTILS_OK) return rc;
    }
    return posv_mixed_run(n, nrhs, A, lda, strideA, B, ldb, strideB, X, ldx, strideX, tol, max_iter, iters, info,
                          work, batch, stream);
}

}  // extern "C"
