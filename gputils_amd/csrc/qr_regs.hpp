// qr_regs.hpp -- Householder QR with the columns held in registers, and the
// entry points of the kernels built on it (qr_regs.hip).
#pragma once

#include "common.hpp"
#include "householder.hpp"

namespace gputils {
namespace qrr {

// Sum over the LPC lanes (16 or 64) that hold one column, in each of them.
template <int LPC, typename T>
__device__ __forceinline__ T lanes_sum(T v) {
    if constexpr (LPC == 16) return hh::row16_sum(v);
    else return wave_sum(v);
}

// Sums over the wavefront of up to four values at once: v_permlane32_swap and
// v_permlane16_swap leave value i's partial sums in 16-lane row i with one
// addition per pair of values, then four row steps finish all of them; lane
// 16 i is value i's sum.  10 additions and swaps for four values, where each
// alone takes 6 steps of two or three instructions.  A value's additions are
// the same whatever it shares the registers with.
__device__ __forceinline__ float swap_add32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double swap_add32(double a, double b) {
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b) {
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
}
template <int N, typename T>
__device__ __forceinline__ void wave_sums(T (&w)[N]) {
    static_assert(N >= 1 && N <= 4, "at most four values");
    // rows 0, 1, 2, 3 of the result: values 0, 2, 1, 3
    const T lo = swap_add32(w[0], w[N > 1 ? 1 : 0]);
    const T hi = N > 2 ? swap_add32(w[N > 2 ? 2 : 0], w[N > 3 ? 3 : N > 2 ? 2 : 0]) : lo;
    const T s = hh::row16_sum(swap_add16(lo, hi));
    constexpr int kLane[4] = {0, 32, 16, 48};
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = readlane(s, kLane[i]);
}

// The reflector scalars without the square root and divisions of
// hh::reflector_scalars: they are on the chain of every column (in FP64 two
// divisions and a square root are about 400 cycles).  FP64: rsq with a
// third-order step, rcp with two Newton steps, and one residual correction
// of the norm and of tau = |alpha - beta| / norm, so that all three are
// rounded as the exact ones are (the errors against 64 bits stay the same).
// FP32 data form them in FP64 with one step each, and round once.
__device__ __forceinline__ void scalars(double alpha, double sq, double &beta, double &tau, double &scale) {
    const double s2 = fma(alpha, alpha, sq);
    const double r = __builtin_amdgcn_rsq(s2);
    const double e = fma(-(s2 * r), r, 1.0);
    const double q = fma(r * e, fma(0.375, e, 0.5), r);  // 1 / norm
    double norm = s2 * q;
    norm = fma(fma(-norm, norm, s2), 0.5 * q, norm);
    const double ad = fabs(alpha) + norm;  // |alpha - beta|
    double inv = __builtin_amdgcn_rcp(ad);
    inv = fma(inv, fma(-ad, inv, 1.0), inv);
    inv = fma(inv, fma(-ad, inv, 1.0), inv);
    tau = ad * q;
    tau = fma(fma(-tau, norm, ad), q, tau);
    beta = (alpha >= 0.0) ? -norm : norm;
    scale = (alpha >= 0.0) ? inv : -inv;
}

// Columns of an m x ntot matrix (m <= LPC * KR, ntot <= NW * 64 / LPC * SL)
// spread over the registers of NW wavefronts: a column belongs to a group
// of LPC lanes (16: four columns per wavefront and slot, 64: one), lane l of
// the group holds its rows l + LPC k, k < KR (zeros past m).  Column c is
// owned by wavefront c % NW, so consecutive columns are formed by different
// wavefronts.  LPC = 16 makes a reduction four steps for four columns; 64
// takes less registers for the reflector that everybody holds, and is for
// the taller matrices.
// NMAX bounds the reflectors, n.  The unit entry of a reflector stays out of the
// lanes' chains, and its product joins the dot product after the reduction:
// it is the largest term, and partial sums that hold it round at its size
// (error against 64 bits of 2500 FP32 systems of 65 to 128 rows 6 % larger).
// NMAX = 0 leaves it in them, for a caller whose errors are set elsewhere.
template <typename T, typename ACC, typename DOT, int LPC, int NW, int KR, int SL, int NMAX = NW * (kWave / LPC) * SL>
struct RegQr {
    static constexpr int kGroups = kWave / LPC;      // columns of one slot of a wavefront
    static constexpr int kCols = NW * kGroups * SL;  // columns held
    static constexpr int kSlots = SL;
    static constexpr int kRows = LPC * KR;
    static constexpr int kUnit = (NMAX + LPC - 1) / LPC < KR ? (NMAX + LPC - 1) / LPC : KR;  // k of row j < kUnit
    static constexpr int kV = 2 * kRows;  // LDS elements of the reflector buffers
    T x[SL][KR];
    int lane, wave, g, l;

    __device__ __forceinline__ RegQr()
        : lane(threadIdx.x & 63), wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), g((threadIdx.x & 63) / LPC),
          l(threadIdx.x & (LPC - 1)) {}
    __device__ __forceinline__ int col(int q) const { return wave + NW * (g + kGroups * q); }
    // first and last column of slot q in this wavefront (uniform)
    __device__ __forceinline__ int first(int q) const { return wave + NW * kGroups * q; }
    __device__ __forceinline__ int last(int q) const { return wave + NW * (kGroups - 1 + kGroups * q); }

    // slot q <- column src of m rows (zeros where !ok); every lane loads a
    // valid element, so that the loads of a column are in flight together
    template <typename S>
    __device__ __forceinline__ void load(int q, const S *src, int m, bool ok) {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int i = l + LPC * k;
            x[q][k] = (T)src[i < m ? i : m - 1];
        }
#pragma unroll
        for (int k = 0; k < KR; ++k)
            if (!(ok && l + LPC * k < m)) x[q][k] = T(0);
    }
    __device__ __forceinline__ void clear(int q) {
#pragma unroll
        for (int k = 0; k < KR; ++k) x[q][k] = T(0);
    }
    __device__ __forceinline__ void store(int q, T *dst, int m, bool ok) const {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int i = l + LPC * k;
            if (ok && i < m) dst[i] = x[q][k];
        }
    }

    // Reflector of column c (this wavefront's slot q): the column becomes
    // [R; beta; v], vb the vector [0 .. 0, 0, v] without its unit entry (with
    // it for kUnit = 0), *s_tau and tau[c] its scalar.
    __device__ __forceinline__ void reflect(T (&xc)[KR], int c, T *vb, T *s_tau, T *tau) {
        const int go = (c / NW) % kGroups;
        T asel = xc[0];
#pragma unroll
        for (int k = 1; k < KR; ++k)
            if (k == c / LPC) asel = xc[k];
        const ACC alpha = (ACC)readlane(asel, go * LPC + c % LPC);
        ACC s0 = ACC(0), s1 = ACC(0);
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const ACC e = (l + LPC * k > c) ? (ACC)xc[k] : ACC(0);
            if (k & 1) s1 = fma(e, e, s1);
            else s0 = fma(e, e, s0);
        }
        const ACC sq = lanes_sum<LPC>(s0 + s1);
        double beta, t, sc;
        if constexpr (sizeof(T) == 8) scalars((double)alpha, (double)sq, beta, t, sc);
        else hh::reflector_scalars<float, double>((double)alpha, (double)sq, beta, t, sc);
        if (sq == ACC(0)) {  // H = I (dlarfg with x = 0): the column stays as it is
            beta = (double)alpha;
            t = 0.0 * fabs((double)alpha);  // NaN for a column that has met an infinity or a NaN
            sc = 1.0;
        }
        const T scale = (T)sc;
        if (g == go) {
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const int i = l + LPC * k;
                const T v = xc[k] * scale;
                vb[i] = (i > c) ? v : ((kUnit == 0 && i == c) ? T(1) : T(0));
                xc[k] = (i > c) ? v : ((i == c) ? (T)beta : xc[k]);
            }
            if (l == 0) {
                *s_tau = (T)t;
                tau[c] = (T)t;
            }
        }
    }

    // row j of this lane's column
    __device__ __forceinline__ T row_of(const T (&xc)[KR], int j) const {
        if constexpr (kUnit == 0) return T(0);
        T xs = xc[0];
#pragma unroll
        for (int k = 1; k < kUnit; ++k)
            if (k == j / LPC) xs = xc[k];  // uniform
        if constexpr (LPC == 64) return readlane(xs, j & 63);
        else return __shfl(xs, (lane & 48) | (j & 15), kWave);
    }
    // entry k of the whole reflector of column j
    __device__ __forceinline__ T whole(const T (&vr)[KR], int k, int j) const {
        return (k < kUnit && l + LPC * k == j) ? T(1) : vr[k];
    }

    // x_q -= (t v . x_q) v for the columns right of column j in slots Q0 ..
    // Q1 - 1 but slot `skip` (uniform; SL for none): the slots' dot products,
    // their reductions and their updates run side by side
    template <int Q0, int Q1>
    __device__ __forceinline__ void update(int skip, int j, int ntot, const T (&vr)[KR], T t) {
        DOT w[Q1 - Q0];
        T xj[Q1 - Q0];
#pragma unroll
        for (int q = Q0; q < Q1; ++q) xj[q - Q0] = row_of(x[q], j);
#pragma unroll
        for (int q = Q0; q < Q1; ++q) {
            DOT w0 = DOT(0), w1 = DOT(0);
#pragma unroll
            for (int k = 0; k < KR; k += 2) {
                w0 = fma((DOT)vr[k], (DOT)x[q][k], w0);
                if (k + 1 < KR) w1 = fma((DOT)vr[k + 1], (DOT)x[q][k + 1], w1);
            }
            w[q - Q0] = w0 + w1;
        }
        if constexpr (LPC == 64) wave_sums(w);
#pragma unroll
        for (int q = Q0; q < Q1; ++q)
            w[q - Q0] = (DOT)t * ((LPC == 64 ? w[q - Q0] : hh::row16_sum(w[q - Q0])) + (DOT)xj[q - Q0]);
#pragma unroll
        for (int q = Q0; q < Q1; ++q) {
            const int c = col(q);
            if (c > j && c < ntot && q != skip) {
#pragma unroll
                for (int k = 0; k < KR; ++k) x[q][k] = fma(-(T)w[q - Q0], whole(vr, k, j), x[q][k]);
            }
        }
    }
    // the same for all slots but those that hold nothing right of column j
    // (uniform): few slots drop out one by one from the left, many in fours
    template <int Q0 = 0>
    __device__ __forceinline__ void update_all(int skip, int j, int ntot, const T (&vr)[KR], T t) {
        if constexpr (SL <= 3) {
            if constexpr (Q0 < SL) {
                if (last(Q0) > j) update<Q0, SL>(skip, j, ntot, vr, t);
                else update_all<Q0 + 1>(skip, j, ntot, vr, t);
            }
        } else if constexpr (Q0 < SL) {
            constexpr int Q1 = Q0 + 4 < SL ? Q0 + 4 : SL;
            if (last(Q1 - 1) > j && first(Q0) < ntot) update<Q0, Q1>(skip, j, ntot, vr, t);
            update_all<Q1>(skip, j, ntot, vr, t);
        }
    }
    // one slot (the owner's next column)
    __device__ __forceinline__ void update_one(T (&xc)[KR], int c, int j, const T (&vr)[KR], T t) {
        const T xj = row_of(xc, j);
        DOT w0 = DOT(0), w1 = DOT(0);
#pragma unroll
        for (int k = 0; k < KR; k += 2) {
            w0 = fma((DOT)vr[k], (DOT)xc[k], w0);
            if (k + 1 < KR) w1 = fma((DOT)vr[k + 1], (DOT)xc[k + 1], w1);
        }
        DOT w[1] = {w0 + w1};
        if constexpr (LPC == 64) wave_sums(w);
        else w[0] = hh::row16_sum(w[0]);
        const T tw = (T)((DOT)t * (w[0] + (DOT)xj));
        if (c > j) {
#pragma unroll
            for (int k = 0; k < KR; ++k) xc[k] = fma(-tw, whole(vr, k, j), xc[k]);
        }
    }

    // Factorises the first n of ntot columns; the others receive every
    // reflector (a right-hand side ends as Q^T b).  vbuf: kV elements and
    // s_tau two of LDS; tau: n values, LDS or global.  Per column: the
    // reflector is read from LDS, the owner of the next column brings that
    // one up to date and forms the next reflector, the others update what
    // they hold; one barrier.  The owner's other columns wait until after the
    // barrier, off the chain.  Ends with a barrier.
    __device__ __forceinline__ void factor(int n, int ntot, T *vbuf, T *s_tau, T *tau) {
        if (wave == 0) reflect(x[0], 0, vbuf, s_tau, tau);
        __syncthreads();
        T vr[KR], t = T(0);
        int late = SL;  // slot formed in the last step: the others wait for its reflector's update
#pragma unroll
        for (int k = 0; k < KR; ++k) vr[k] = T(0);
#pragma unroll 1
        for (int j = 0; j < n; ++j) {
            if (late < SL) {  // uniform; vr and t are still the last step's
                update_all(late, j - 1, ntot, vr, t);
                late = SL;
            }
            const T *v = vbuf + (j & 1) * kRows;
#pragma unroll
            for (int k = 0; k < KR; ++k) vr[k] = v[l + LPC * k];
            t = s_tau[j & 1];
            const int c1 = j + 1;
            if (c1 < n && wave == c1 % NW) {  // uniform
                late = c1 / (NW * kGroups);
#pragma unroll
                for (int q = 0; q < SL; ++q)
                    if (q == late) {
                        update_one(x[q], col(q), j, vr, t);  // columns past ntot hold zeros
                        reflect(x[q], c1, vbuf + (c1 & 1) * kRows, s_tau + (c1 & 1), tau);
                    }
            } else {
                update_all(SL, j, ntot, vr, t);
            }
            __syncthreads();
        }
    }
};

// Rows of the tallest matrices, and order of the largest triangles, that the
// register kernels take.
constexpr int kMaxRows = 1024;
constexpr int kMaxTri = 512;

// Householder QR of the m x n matrices (m <= kMaxRows) in LAPACK storage.
// tau may be NULL (not stored).
template <typename T>
int geqrf(int64_t m, int64_t n, T *A, int64_t lda, int64_t strideA, T *tau, int64_t strideTau, int *info,
          int64_t batch, hipStream_t st);
// Least squares, m <= kMaxRows and n <= kMaxTri.
template <typename T>
int gels(int64_t m, int64_t n, int64_t nrhs, T *A, int64_t lda, int64_t strideA, T *B, int64_t ldb, int64_t strideB,
         int *info, int64_t batch, hipStream_t st);
// The first mout rows of C <- Q^T C or Q C, m <= kMaxRows.  tau NULL: formed
// from the reflectors.
template <typename T>
int ormqr(int trans, int64_t m, int64_t mout, int64_t ncols, int64_t k, const T *A, int64_t lda, int64_t strideA,
          const T *tau, int64_t strideTau, T *C, int64_t ldc, int64_t strideC, int64_t batch, hipStream_t st);
// B <- R^{-1} B, n <= kMaxTri.
template <typename T>
int trsm_upper(int64_t n, int64_t nrhs, const T *R, int64_t ldr, int64_t strideR, T *B, int64_t ldb, int64_t strideB,
               int64_t batch, hipStream_t st);

}  // namespace qrr
}  // namespace gputils
