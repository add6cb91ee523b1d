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
template <typename T, typename ACC, typename DOT, int LPC, int NW, int KR, int SL>
struct RegQr {
    static constexpr int kGroups = kWave / LPC;      // columns of one slot of a wavefront
    static constexpr int kCols = NW * kGroups * SL;  // columns held
    static constexpr int kRows = LPC * KR;
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
    __device__ __forceinline__ void store(int q, T *dst, int m, bool ok) const {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int i = l + LPC * k;
            if (ok && i < m) dst[i] = x[q][k];
        }
    }

    // Reflector of column c (this wavefront's slot q): the column becomes
    // [R; beta; v], vb the whole vector [0 .. 0, 1, v], *s_tau and tau[c] its
    // scalar.
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
            t = 0.0;
            sc = 1.0;
        }
        const T scale = (T)sc;
        if (g == go) {
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const int i = l + LPC * k;
                const T v = xc[k] * scale;
                vb[i] = (i > c) ? v : ((i == c) ? T(1) : T(0));
                xc[k] = (i > c) ? v : ((i == c) ? (T)beta : xc[k]);
            }
            if (l == 0) {
                *s_tau = (T)t;
                tau[c] = (T)t;
            }
        }
    }

    // x_q -= (t v . x_q) v for the columns right of column j in slots Q0 ..
    // SL - 1 but slot `skip` (uniform; SL for none): the slots' dot products,
    // their reductions and their updates run side by side
    template <int Q0>
    __device__ __forceinline__ void update(int skip, int j, int ntot, const T (&vr)[KR], T t) {
        DOT w[SL];
#pragma unroll
        for (int q = Q0; q < SL; ++q) {
            DOT w0 = DOT(0), w1 = DOT(0);
#pragma unroll
            for (int k = 0; k < KR; k += 2) {
                w0 = fma((DOT)vr[k], (DOT)x[q][k], w0);
                if (k + 1 < KR) w1 = fma((DOT)vr[k + 1], (DOT)x[q][k + 1], w1);
            }
            w[q] = w0 + w1;
        }
#pragma unroll
        for (int q = Q0; q < SL; ++q) w[q] = (DOT)t * lanes_sum<LPC>(w[q]);
#pragma unroll
        for (int q = Q0; q < SL; ++q) {
            const int c = col(q);
            if (c > j && c < ntot && q != skip) {
#pragma unroll
                for (int k = 0; k < KR; ++k) x[q][k] = fma(-(T)w[q], vr[k], x[q][k]);
            }
        }
    }
    // one slot (the owner's next column)
    __device__ __forceinline__ void update_one(T (&xc)[KR], int c, int j, const T (&vr)[KR], T t) {
        DOT w0 = DOT(0), w1 = DOT(0);
#pragma unroll
        for (int k = 0; k < KR; k += 2) {
            w0 = fma((DOT)vr[k], (DOT)xc[k], w0);
            if (k + 1 < KR) w1 = fma((DOT)vr[k + 1], (DOT)xc[k + 1], w1);
        }
        const T tw = (T)((DOT)t * lanes_sum<LPC>(w0 + w1));
        if (c > j) {
#pragma unroll
            for (int k = 0; k < KR; ++k) xc[k] = fma(-tw, vr[k], xc[k]);
        }
    }

    // Factorises the first n of ntot columns; the others receive every
    // reflector (a right-hand side ends as Q^T b).  vbuf: kV elements and
    // s_tau two of LDS; tau: n values, LDS or global.  Per column: the
    // reflector is read from LDS, the owner of the next column brings that
    // one up to date first and forms the next reflector, the others update
    // what they hold; one barrier.  Ends with a barrier.
    __device__ __forceinline__ void factor(int n, int ntot, T *vbuf, T *s_tau, T *tau) {
        if (wave == 0) reflect(x[0], 0, vbuf, s_tau, tau);
        __syncthreads();
#pragma unroll 1
        for (int j = 0; j < n; ++j) {
            const T *v = vbuf + (j & 1) * kRows;
            T vr[KR];
#pragma unroll
            for (int k = 0; k < KR; ++k) vr[k] = v[l + LPC * k];
            const T t = s_tau[j & 1];
            const int c1 = j + 1;
            const bool own = c1 < n && wave == c1 % NW;  // uniform
            const int q1 = own ? c1 / (NW * kGroups) : SL;
            if (own) {
#pragma unroll
                for (int q = 0; q < SL; ++q)
                    if (q == q1) {
                        update_one(x[q], col(q), j, vr, t);  // columns past ntot hold zeros
                        reflect(x[q], c1, vbuf + (c1 & 1) * kRows, s_tau + (c1 & 1), tau);
                    }
            }
            // slots whose columns are all factorised drop out from the left
            constexpr int kQ = SL >= 4 ? SL / 4 : 1;
            if (last(kQ - 1) > j) update<0>(q1, j, ntot, vr, t);
            else if (SL > kQ && last(2 * kQ - 1 < SL ? 2 * kQ - 1 : 0) > j) update<kQ < SL ? kQ : 0>(q1, j, ntot, vr, t);
            else if (SL > 2 * kQ && last(3 * kQ - 1 < SL ? 3 * kQ - 1 : 0) > j)
                update<2 * kQ < SL ? 2 * kQ : 0>(q1, j, ntot, vr, t);
            else if (SL > 3 * kQ) update<3 * kQ < SL ? 3 * kQ : 0>(q1, j, ntot, vr, t);
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
