// qr_regs.hip -- batched Householder QR, least squares and Q application with
// the columns in registers, for gfx950 (see RegQr in qr_regs.hpp).
//
// The column steps of a QR are a chain: reflector, dot products, update.
// Streaming the columns from LDS or global memory for every step made a
// step 1.5 to 40 us; here a column is loaded once, stays in the registers of
// the lanes that own it, and only the reflector goes through LDS.  What
// bounds a step now is the chain reflector -> dot product -> update -> next
// reflector (about 0.6 us in FP32, 1 us in FP64) and, with many matrices,
// instruction issue (VALU issue in 65 % of the cycles of 1024 least-squares
// systems).  Before -> now: least squares of 1024 FP32 100 x 30 systems 91 -> 35
// us; QR of one FP64 600 x 150 matrix 6320 -> 250 us, its 150 columns of Q
// 10357 -> 64 us.
#include <algorithm>

#include "qr_regs.hpp"

namespace gputils {
namespace qrr {

// Back substitution R y = c by one wavefront: lane i holds rows i + 64 u of c
// and the reciprocals of R's diagonal, column k - 1 of R (LDS, ld ldr) is
// read while step k runs.  Where one has no normal reciprocal it divides.
template <typename T, int NR>
__device__ __forceinline__ void trsv_regs(const T *R, int ldr, int n, T *c) {
    const int lane = threadIdx.x & 63;
    T cv[NR], di[NR], rk[NR];
    bool divide = false;
#pragma unroll
    for (int u = 0; u < NR; ++u) {
        const int i = lane + kWave * u;
        cv[u] = (i < n) ? c[i] : T(0);
        di[u] = (i < n) ? R[i + i * ldr] : T(1);
        divide = divide || !hh::has_reciprocal(di[u]);
        di[u] = T(1) / di[u];
        rk[u] = (i < n) ? R[i + (n - 1) * ldr] : T(0);
    }
    if (__builtin_expect(__any(divide), 0)) {
        hh::trsv_upper<T>(R, ldr, n, c);
        return;
    }
#pragma unroll 1
    for (int k = n - 1; k >= 0; --k) {
        T rn[NR];
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            const int i = lane + kWave * u;
            rn[u] = (i < k) ? R[i + (k - 1) * ldr] : T(0);
        }
        T cs = cv[0], ds = di[0];
#pragma unroll
        for (int u = 1; u < NR; ++u)
            if (k >= kWave * u) {  // uniform
                cs = cv[u];
                ds = di[u];
            }
        const T ck = readlane(cs, k & 63) * readlane(ds, k & 63);
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            const int i = lane + kWave * u;
            cv[u] = (i == k) ? ck : ((i < k) ? fma(-rk[u], ck, cv[u]) : cv[u]);
            rk[u] = rn[u];
        }
    }
#pragma unroll
    for (int u = 0; u < NR; ++u) {
        const int i = lane + kWave * u;
        if (i < n) c[i] = cv[u];
    }
}

// The first n rows of Q^T b by one wavefront, lane i holding rows i + 64 u of b:
// a reflector takes and changes the rows from its own on and no others, and H = I
// none, so that an infinity or a NaN reaches no row that it should not.
template <typename T, int U>
__device__ __forceinline__ void qtb_plain(const T *A, int64_t lda, int m, int n, const T *tau, const T *b, T *c) {
    const int lane = threadIdx.x & 63;
    T y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) y[u] = (lane + kWave * u < m) ? b[lane + kWave * u] : T(0);
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
        const T t = tau[j];
        if (t == T(0)) continue;
        const T *v = A + (int64_t)j * lda;
        T w = T(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = lane + kWave * u;
            if (i >= j && i < m) w = fma(i == j ? T(1) : v[i], y[u], w);
        }
        w = t * wave_sum(w);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = lane + kWave * u;
            if (i >= j && i < m) y[u] = fma(-w, i == j ? T(1) : v[i], y[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (lane + kWave * u < n) c[lane + kWave * u] = y[u];
    hh::wave_sync();
}

// For reflectors whose scalars will be formed again from v (ormqr_regs_kernel),
// where |v|^2 = 0 stands for H = I.  A tail so small beside alpha that its square
// underflows has tau = 2 and beta = -alpha all the same: the first entry of such a
// v becomes kMark, whose square is a normal number and whose effect lies far below
// the type's rounding.  Reads back what the workgroup has just stored, and that of
// reflectors with tau = 2 only, so that it costs the others nothing.
template <typename T, int NW>
__device__ __forceinline__ void mark_tails(T *A, int64_t lda, int m, int n, const T *tau) {
    constexpr T kMark = sizeof(T) == 8 ? T(0x1p-450) : T(0x1p-60);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    for (int c = wave; c < n; c += NW) {
        if (!(tau[c] > T(1.999))) continue;
        T *v = A + (int64_t)c * lda;
        T s = T(0);
        for (int i = c + 1 + lane; i < m; i += kWave) s = fma(v[i], v[i], s);
        if (wave_sum(s) == T(0) && lane == 0) v[c + 1] = kMark;
    }
}

// Wavefronts per SIMD to leave registers for: what the column steps alone take,
// by the 32-bit words of the columns.  Left to itself the compiler gives the
// rare path below some more, and 8192 FP32 100 x 30 factorisations (66 registers
// where 64 fit) take 153 us instead of 147.
constexpr int qr_waves(int words) {
    return words <= 14 ? 8 : words <= 16 ? 7 : words <= 20 ? 6 : words <= 24 ? 5 : words <= 32 ? 4 : words <= 48 ? 3 : words <= 64 ? 2 : 1;
}

// QR of one matrix per workgroup, and with nrhs > 0 the least-squares
// solution: the right-hand sides ride along as columns n .. n + nrhs - 1, so
// the factorisation leaves Q^T b; R and those go to LDS and one wavefront
// per right-hand side substitutes back.  tau may be NULL.
// In the registers the rows above a reflector meet zeros of it, through which
// infinities and NaNs reach rows that the reflector does not.  A column that
// has met one is NaN throughout and so is its scalar: the matrix, still as it
// was in memory, is then factorised again there (hh::hqr_plain).
template <typename T, int LPC, int NW, int KR, int SL>
__global__ __launch_bounds__(NW *kWave) __attribute__((amdgpu_waves_per_eu(
    qr_waves(KR *SL *(int)sizeof(T) / 4) > NW / 4 ? qr_waves(KR *SL *(int)sizeof(T) / 4) : (NW + 3) / 4))) void qr_regs_kernel(int m, int n, int nrhs, T *A, int64_t lda,
                                                            int64_t strideA, T *B, int64_t ldb, int64_t strideB,
                                                            T *tau, int64_t strideTau, int *info, int64_t batch) {
    using Q = RegQr<T, T, T, LPC, NW, KR, SL>;
    __shared__ T vbuf[Q::kV];
    __shared__ T s_tau[2];
    __shared__ T taus[Q::kCols];
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_regs[];  // n x (n + nrhs) with nrhs > 0
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    T *a = A + b * strideA;
    T *bb = B + b * strideB;
    Q qr;
#pragma unroll
    for (int q = 0; q < SL; ++q) {
        const int c = qr.col(q);
        const T *src = (c >= n && c < n + nrhs) ? bb + (int64_t)(c - n) * ldb : a + (int64_t)(c < n ? c : 0) * lda;
        qr.load(q, src, m, c < n + nrhs);
    }
    qr.factor(n, n + nrhs, vbuf, s_tau, taus);
    bool odd = false;
    for (int i = qr.lane; i < n; i += kWave) odd = odd || !__builtin_isfinite(taus[i]);
    if (__builtin_expect(__any(odd), 0)) {  // the same in every wavefront
        __syncthreads();  // all have read taus before it is formed again
        hh::hqr_plain<T, T, NW>(a, lda, m, n, taus, s_tau);
        if (tau != nullptr)
            for (int i = threadIdx.x; i < n; i += NW * kWave) tau[b * strideTau + i] = taus[i];
        if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
        for (int r = qr.wave; r < nrhs; r += NW) {
            T *rhs = bb + (int64_t)r * ldb, *c = reinterpret_cast<T *>(dyn_regs) + r * n;
            qtb_plain<T, (Q::kRows + kWave - 1) / kWave>(a, lda, m, n, taus, rhs, c);
            hh::trsv_upper<T>(a, lda, n, c);
            for (int i = qr.lane; i < n; i += kWave) rhs[i] = c[i];
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < SL; ++q) qr.store(q, a + (int64_t)qr.col(q) * lda, m, qr.col(q) < n);
    if (tau != nullptr)
        for (int i = threadIdx.x; i < n; i += NW * kWave) tau[b * strideTau + i] = taus[i];
    if (threadIdx.x == 0 && info != nullptr) info[b] = 0;
    if (nrhs == 0) {
        if (tau == nullptr) mark_tails<T, NW>(a, lda, m, n, taus);  // uniform
        return;
    }
    T *R = reinterpret_cast<T *>(dyn_regs);
    const int ldr = n | 1;
#pragma unroll
    for (int q = 0; q < SL; ++q) qr.store(q, R + qr.col(q) * ldr, n, qr.col(q) < n + nrhs);
    __syncthreads();
    for (int r = qr.wave; r < nrhs; r += NW) {
        T *c = R + (n + r) * ldr;
        bool spread = false;  // an infinity or a NaN in Q^T b
        for (int i = qr.lane; i < n; i += kWave) spread = spread || !__builtin_isfinite(c[i]);
        if (__builtin_expect(__any(spread), 0)) qtb_plain<T, (Q::kRows + kWave - 1) / kWave>(a, lda, m, n, taus, bb + (int64_t)r * ldb, c);
        if (n <= kWave) trsv_regs<T, 1>(R, ldr, n, c);
        else trsv_regs<T, 2>(R, ldr, n, c);
        hh::wave_sync();
        for (int i = qr.lane; i < n; i += kWave) bb[i + (int64_t)r * ldb] = c[i];
    }
}

// C <- Q^T C (trans) or Q C, Q from k reflectors.  A wavefront holds SL
// columns of C in registers (rows lane + 64 u, u < R) for all the
// reflectors; the workgroup stages kChunk of them at a time in LDS, as
// vectors [0 .. 0, 0, v] without the unit entry, the next ones already on
// their way.  Bound by the chain of a reflector (its LDS reads, one wave reduction, the update), so
// few columns go one to a wavefront over as many workgroups as there are;
// batches that fill the chip take four.  tau NULL: the scalar is formed from
// the vector, tau = 2 / (1 + |v|^2), or 0 for |v|^2 = 0 (H = I): least squares has
// no room to keep it between launches, and mark_tails sees to it that no
// other reflector has |v|^2 = 0.  Columns that come out with an infinity or a
// NaN are done again through LDS (see qr_regs_kernel).  Only the first mout rows of C are
// written (least squares leaves the rest of b as it was).
constexpr int kOrmThreads = 256;
constexpr int kOrmWaves = kOrmThreads / kWave;
constexpr int kChunk = 8;
template <typename T, int R, int SL>
__global__ __launch_bounds__(kOrmThreads) void ormqr_regs_kernel(int trans, int m, int mout, int ncols, int k, const T *A,
                                                                 int64_t lda, int64_t strideA, const T *tau,
                                                                 int64_t strideTau, T *C, int64_t ldc,
                                                                 int64_t strideC, int64_t batch) {
    constexpr int kRows = kWave * R;
    __shared__ T V[kChunk][kRows];
    __shared__ T s_tau[kChunk];
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T *a = A + b * strideA;
    const T *tb = tau + (tau != nullptr ? b * strideTau : 0);
    T *cb = C + b * strideC;
    const int c0 = (blockIdx.y * kOrmWaves + wave) * SL;
    T x[SL][R];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        const T *src = cb + (int64_t)(c0 + s < ncols ? c0 + s : 0) * ldc;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int i = lane + kWave * u;
            x[s][u] = src[i < m ? i : m - 1];
        }
#pragma unroll
        for (int u = 0; u < R; ++u)
            if (lane + kWave * u >= m) x[s][u] = T(0);
    }
    // chunk q of reflectors in the order they are applied (aligned to kChunk):
    // entry e of its ne(q) is reflector refl(q, e); wavefront w stages entries
    // w and w + 4
    const int chunks = (k + kChunk - 1) / kChunk;
    auto base = [&](int q) { return (trans ? q : chunks - 1 - q) * kChunk; };
    auto count = [&](int q) { return k - base(q) < kChunk ? k - base(q) : kChunk; };
    auto refl = [&](int q, int e) { return trans ? base(q) + e : base(q) + count(q) - 1 - e; };
    // The rows of a chunk's unit entries lie in one block of 64: it and block 0
    // change places in the registers and in V, so that the unit entry is always
    // in slot 0.  Its product joins the dot product after the reduction (see
    // RegQr).  A 600 x 150 FP64 QR, solution and Q took 405 us so, as with the
    // entry in the lanes' sums, and 458 with the row's register selected in
    // every step.
    int head = 0;  // block in slot 0
    auto swap0 = [&](int u0) {
#pragma unroll
        for (int u = 1; u < R; ++u) {
            const bool take = u == u0;  // uniform; selects, as a branch would index x (scratch)
#pragma unroll
            for (int s = 0; s < SL; ++s) {
                const T y = x[s][0], z = x[s][u];
                x[s][0] = take ? z : y;
                x[s][u] = take ? y : z;
            }
        }
    };
    constexpr int kPer = kChunk / kOrmWaves;
    T nv[kPer][R];
    auto fetch = [&](int q) {
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            const int e = wave + kOrmWaves * p;
            const int j = e < count(q) ? refl(q, e) : 0;
            const T *col = a + (int64_t)j * lda;
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const int i = lane + kWave * u;
                nv[p][u] = col[i < m ? i : m - 1];
            }
        }
    };
    fetch(0);
#pragma unroll 1
    for (int q = 0; q < chunks; ++q) {
        const int ne = count(q), ju = base(q) / kWave;
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            const int e = wave + kOrmWaves * p;
            const int j = refl(q, e);
            T vv = T(0);
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const int i = lane + kWave * u;
                const T v = (i > j && i < m) ? nv[p][u] : T(0);
                vv = fma(v, v, vv);
                V[e][lane + kWave * (u == ju ? 0 : u == 0 ? ju : u)] = v;
            }
            if (tau == nullptr) {  // uniform
                vv = wave_sum(vv);
                if (lane == 0) s_tau[e] = (vv == T(0)) ? T(0) : T(2) / (T(1) + vv);
            }
        }
        if (tau != nullptr && (int)threadIdx.x < ne) s_tau[threadIdx.x] = tb[refl(q, threadIdx.x)];
        __syncthreads();
        if (q + 1 < chunks) fetch(q + 1);
        if (ju != head) {  // uniform
            swap0(head);
            swap0(ju);
            head = ju;
        }
        if (c0 < ncols) {  // uniform
#pragma unroll 1
            for (int e = 0; e < ne; ++e) {
                const int jl = refl(q, e) & (kWave - 1);
                T vr[R];
#pragma unroll
                for (int u = 0; u < R; ++u) vr[u] = V[e][lane + kWave * u];
                const T t = s_tau[e];
                T w[SL], xj[SL];
#pragma unroll
                for (int s = 0; s < SL; ++s) xj[s] = readlane(x[s][0], jl);
#pragma unroll
                for (int s = 0; s < SL; ++s) {
                    T w0 = T(0), w1 = T(0);
#pragma unroll
                    for (int u = 0; u < R; u += 2) {
                        w0 = fma(vr[u], x[s][u], w0);
                        if (u + 1 < R) w1 = fma(vr[u + 1], x[s][u + 1], w1);
                    }
                    w[s] = w0 + w1;
                }
                if (lane == jl) vr[0] = T(1);
#pragma unroll
                for (int s = 0; s < SL; ++s) w[s] = t * (wave_sum(w[s]) + xj[s]);
                if (t != T(0)) {  // H = I stays out of C
#pragma unroll
                    for (int s = 0; s < SL; ++s)
#pragma unroll
                        for (int u = 0; u < R; ++u) x[s][u] = fma(-w[s], vr[u], x[s][u]);
                }
            }
        }
        __syncthreads();
    }
    swap0(head);
    bool odd = false;
#pragma unroll
    for (int s = 0; s < SL; ++s) odd = odd || !__builtin_isfinite(x[s][0]);
    if (__builtin_expect(__any(odd), 0)) {
        T *c = V[wave];  // this wavefront's own row; the last reflectors are past
        for (int s = c0; s < c0 + SL && s < ncols; ++s) {
            T *dst = cb + (int64_t)s * ldc;
            for (int i = lane; i < m; i += kWave) c[i] = dst[i];
            hh::wave_sync();
            for (int e = 0; e < k; ++e) {
                const int j = trans ? e : k - 1 - e;
                const T *v = a + (int64_t)j * lda;
                T t;
                if (tau != nullptr) {
                    t = tb[j];
                } else {
                    t = T(0);
                    for (int i = j + 1 + lane; i < m; i += kWave) t = fma(v[i], v[i], t);
                    t = wave_sum(t);
                    t = (t == T(0)) ? T(0) : T(2) / (T(1) + t);
                }
                hh::apply_reflector_vec<T, T>(v, m, j, t, c);
            }
            for (int i = lane; i < mout; i += kWave) dst[i] = c[i];
            hh::wave_sync();
        }
        return;
    }
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        if (c0 + s >= ncols) continue;
        T *dst = cb + (int64_t)(c0 + s) * ldc;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int i = lane + kWave * u;
            if (i < mout) dst[i] = x[s][u];
        }
    }
}

// B <- R^{-1} B, R upper triangular n x n (n <= 64 NU).  A wavefront solves
// one column: lane i holds rows i + 64 u of it and the reciprocals of R's
// diagonal; the workgroup's four share R, staged through LDS 16 columns at a
// time with the next ones on their way.  A step is a broadcast, a product and
// NU FMAs (about 90 cycles), where reading R's column from global memory in
// every step made it 900: n = 150 in FP64, one column, 59 -> 20 us.  Where a
// diagonal entry has no normal reciprocal it divides, with R in memory.
constexpr int kTrsmCols = 16;
template <typename T, int NU>
__global__ __launch_bounds__(kOrmThreads) void trsm_regs_kernel(int n, int nrhs, const T *R, int64_t ldr,
                                                                int64_t strideR, T *B, int64_t ldb, int64_t strideB,
                                                                int64_t batch) {
    constexpr int kRows = kWave * NU;
    __shared__ T S[kTrsmCols][kRows];
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T *r = R + b * strideR;
    const int col = blockIdx.y * kOrmWaves + wave;
    const bool ok = col < nrhs;
    T *x = B + b * strideB + (int64_t)(ok ? col : 0) * ldb;
    T c[NU], di[NU];
    bool divide = false;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int i = lane + kWave * u;
        c[u] = (i < n) ? x[i] : T(0);
        di[u] = (i < n) ? r[i + (int64_t)i * ldr] : T(1);
        divide = divide || !hh::has_reciprocal(di[u]);
        di[u] = T(1) / di[u];
    }
    if (__builtin_expect(__any(divide), 0)) {  // the same in every wavefront
        T *y = S[wave];  // n <= kRows
        if (ok) {
            for (int i = lane; i < n; i += kWave) y[i] = x[i];
            hh::wave_sync();
            hh::trsv_upper<T>(r, ldr, n, y);
            for (int i = lane; i < n; i += kWave) x[i] = y[i];
        }
        return;
    }
    // columns 16 q .. 16 q + 15; wavefront w stages four of them
    constexpr int kPer = kTrsmCols / kOrmWaves;
    T nv[kPer][NU];
    auto fetch = [&](int q) {
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            const int k = kTrsmCols * q + wave * kPer + p;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int i = lane + kWave * u;
                nv[p][u] = r[(i < n ? i : n - 1) + (int64_t)(k < n ? k : n - 1) * ldr];
            }
        }
    };
    constexpr int kPer64 = kWave / kTrsmCols;  // stages of 64 rows
    fetch((n - 1) / kTrsmCols);
#pragma unroll
    for (int u0 = NU - 1; u0 >= 0; --u0) {
#pragma unroll 1
        for (int h = kPer64 - 1; h >= 0; --h) {
            const int q = u0 * kPer64 + h;
            if (kTrsmCols * q >= n) continue;  // uniform
            __syncthreads();
#pragma unroll
            for (int p = 0; p < kPer; ++p)
#pragma unroll
                for (int u = 0; u <= u0; ++u) S[wave * kPer + p][lane + kWave * u] = nv[p][u];
            __syncthreads();
            if (q > 0) fetch(q - 1);
            if (!ok) continue;
#pragma unroll
            for (int e = kTrsmCols - 1; e >= 0; --e) {
                const int kk = kTrsmCols * h + e;  // lane of row k
                if (kWave * u0 + kk >= n) continue;  // uniform
                const T ck = readlane(c[u0], kk) * readlane(di[u0], kk);
#pragma unroll
                for (int u = 0; u < u0; ++u) c[u] = fma(-S[e][lane + kWave * u], ck, c[u]);
                const T s = S[e][lane + kWave * u0];
                c[u0] = (lane == kk) ? ck : ((lane < kk) ? fma(-s, ck, c[u0]) : c[u0]);
            }
        }
    }
    if (ok) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int i = lane + kWave * u;
            if (i < n) x[i] = c[u];
        }
    }
}

// ------------------------------------------------------------ dispatch --
namespace {

// Columns of a panel of the launches-per-panel form: one slot in each of 16
// wavefronts, so that a column step is not bound by what one CU can issue
// (600 x 150 in FP64, factorisation: 256 us with panels of 32 and two slots,
// 249 with 16).
constexpr int kPanel = 16;

// The instantiation for m rows and nt columns, or NULL.  16-lane columns up
// to 256 rows and 128 columns (FP64 of more than 160 rows: 96, where the
// registers end); taller matrices by whole wavefronts, kPanel columns of them,
// which every m <= kMaxRows takes, and whatever is wider in panels.  Several
// slots of whole wavefronts spilled 13 to 100 registers and were 2 to 5 times
// slower than panels for any batch: 128 and 1024 FP32 384 x 80 factorisations
// 281 and 1259 us, in panels 104 and 303.
template <typename T>
struct QrPick {
    void (*kern)(int, int, int, T *, int64_t, int64_t, T *, int64_t, int64_t, T *, int64_t, int *, int64_t) = nullptr;
    int threads = 0;
    int lds = 0;  // static bytes
    template <int LPC, int NW, int KR, int SL>
    void set() {
        kern = qr_regs_kernel<T, LPC, NW, KR, SL>;
        threads = NW * kWave;
        using Q = RegQr<T, T, T, LPC, NW, KR, SL>;
        lds = (int)sizeof(T) * (Q::kV + 2 + Q::kCols);
    }
    template <int KR>
    void set16(int nt) {
        if (nt <= 16) set<16, 2, KR, 2>();
        else if (nt <= 32) set<16, 4, KR, 2>();
        else if (nt <= 48) set<16, 4, KR, 3>();
        else if (nt <= 64) set<16, 8, KR, 2>();
        else if (nt <= 96) set<16, 8, KR, 3>();
        else if constexpr ((int)sizeof(T) * KR < 128) {
            if (nt <= 128) set<16, 16, KR, 2>();
        }
    }
    QrPick(int64_t m, int64_t nt) {
        if (m <= 32) set16<2>((int)nt);
        else if (m <= 64) set16<4>((int)nt);
        else if (m <= 112) set16<7>((int)nt);
        else if (m <= 160) set16<10>((int)nt);
        else if (m <= 256) set16<16>((int)nt);
        else if (nt <= kPanel) {
            if (m <= 384) set<64, 16, 6, 1>();
            else if (m <= 640) set<64, 16, 10, 1>();
            else if (m <= kMaxRows) set<64, 16, 16, 1>();
        }
    }
};

constexpr int kMaxDyn = 128 * 1024;  // of 160 KB; the kernels' own arrays take 17 at most

}  // namespace

template <typename T>
int geqrf(int64_t m, int64_t n, T *A, int64_t lda, int64_t strideA, T *tau, int64_t strideTau, int *info,
          int64_t batch, hipStream_t st) {
    const QrPick<T> whole(m, n);
    if (whole.kern != nullptr) {
        hipLaunchKernelGGL(whole.kern, dim3((unsigned)batch), dim3(whole.threads), 0, st, (int)m, (int)n, 0, A, lda,
                           strideA, A, lda, strideA, tau, strideTau, info, batch);
        return launch_check("qr_regs_kernel");
    }
    // panels of kPanel columns: one workgroup factorises the panel, then its
    // reflectors are applied to the columns right of it by as many workgroups
    // as those need
    for (int64_t j = 0; j < n; j += kPanel) {
        const int64_t w = std::min<int64_t>(kPanel, n - j), rest = n - j - w;
        T *p = A + j + j * lda;
        const QrPick<T> panel(m - j, w);
        hipLaunchKernelGGL(panel.kern, dim3((unsigned)batch), dim3(panel.threads), 0, st, (int)(m - j), (int)w, 0, p,
                           lda, strideA, p, lda, strideA, tau != nullptr ? tau + j : tau, strideTau, info, batch);
        int rc = launch_check("qr_regs_kernel");
        if (rc == GPUTILS_OK && rest > 0)
            rc = ormqr<T>(1, m - j, m - j, rest, w, p, lda, strideA, tau != nullptr ? tau + j : tau, strideTau, p + w * lda, lda,
                          strideA, batch, st);
        if (rc != GPUTILS_OK) return rc;
    }
    return GPUTILS_OK;
}

template <typename T>
int gels(int64_t m, int64_t n, int64_t nrhs, T *A, int64_t lda, int64_t strideA, T *B, int64_t ldb, int64_t strideB,
         int *info, int64_t batch, hipStream_t st) {
    // one launch where R and the right-hand sides fit the LDS
    const QrPick<T> whole(m, n + nrhs);
    const size_t dyn = nrhs > 0 ? sizeof(T) * (size_t)((n | 1) * (n + nrhs)) : 0;
    if (whole.kern != nullptr && n <= 2 * kWave && dyn <= (size_t)kMaxDyn) {
        // the same value from every call: another thread's launch of this kernel
        // may come between this line and the next
        if (whole.lds + dyn > 64 * 1024)
            GPUTILS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(whole.kern),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, kMaxDyn));
        hipLaunchKernelGGL(whole.kern, dim3((unsigned)batch), dim3(whole.threads), dyn, st, (int)m, (int)n, (int)nrhs,
                           A, lda, strideA, B, ldb, strideB, (T *)nullptr, (int64_t)0, info, batch);
        return launch_check("qr_regs_kernel");
    }
    int rc = geqrf<T>(m, n, A, lda, strideA, nullptr, 0, info, batch, st);
    if (rc == GPUTILS_OK && nrhs > 0)
        rc = ormqr<T>(1, m, n, nrhs, n, A, lda, strideA, nullptr, 0, B, ldb, strideB, batch, st);
    if (rc == GPUTILS_OK && nrhs > 0) rc = trsm_upper<T>(n, nrhs, A, lda, strideA, B, ldb, strideB, batch, st);
    return rc;
}

template <typename T>
int ormqr(int trans, int64_t m, int64_t mout, int64_t ncols, int64_t k, const T *A, int64_t lda, int64_t strideA,
          const T *tau, int64_t strideTau, T *C, int64_t ldc, int64_t strideC, int64_t batch, hipStream_t st) {
    // four columns a wavefront once that still gives four wavefronts per SIMD:
    // below it the chain of each reflector is what counts (1024 FP32 100 x 30
    // factors, 30 columns: 40 us, 189 with the column in LDS)
    const bool wide = ncols * batch >= 4 * 4096 && m <= 640;
    const int64_t per = (wide ? 4 : 1) * kOrmWaves;
    for (int64_t c0 = 0; c0 < ncols; c0 += per * 65535) {
        const int64_t nc = std::min<int64_t>(ncols - c0, per * 65535);
        const dim3 grid((unsigned)batch, (unsigned)ceil_div(nc, per));
#define GPUTILS_ORM(RV)                                                                                            \
    hipLaunchKernelGGL((wide ? ormqr_regs_kernel<T, RV, 4> : ormqr_regs_kernel<T, RV, 1>), grid, dim3(kOrmThreads), \
                       0, st, trans, (int)m, (int)mout, (int)nc, (int)k, A, lda, strideA, tau, strideTau, C + c0 * ldc, ldc, \
                       strideC, batch)
        if (m <= 64) GPUTILS_ORM(1);
        else if (m <= 128) GPUTILS_ORM(2);
        else if (m <= 256) GPUTILS_ORM(4);
        else if (m <= 384) GPUTILS_ORM(6);
        else if (m <= 640) GPUTILS_ORM(10);
        else
            hipLaunchKernelGGL((ormqr_regs_kernel<T, 16, 1>), grid, dim3(kOrmThreads), 0, st, trans, (int)m, (int)mout,
                               (int)nc, (int)k, A, lda, strideA, tau, strideTau, C + c0 * ldc, ldc, strideC, batch);
#undef GPUTILS_ORM
        const int rc = launch_check("ormqr_regs_kernel");
        if (rc != GPUTILS_OK) return rc;
    }
    return GPUTILS_OK;
}

template <typename T>
int trsm_upper(int64_t n, int64_t nrhs, const T *R, int64_t ldr, int64_t strideR, T *B, int64_t ldb, int64_t strideB,
               int64_t batch, hipStream_t st) {
    for (int64_t c0 = 0; c0 < nrhs; c0 += kOrmWaves * 65535) {
        const int64_t nc = std::min<int64_t>(nrhs - c0, kOrmWaves * 65535);
        const dim3 grid((unsigned)batch, (unsigned)ceil_div(nc, kOrmWaves));
        auto kern = n <= 64    ? trsm_regs_kernel<T, 1>
                    : n <= 128 ? trsm_regs_kernel<T, 2>
                    : n <= 256 ? trsm_regs_kernel<T, 4>
                               : trsm_regs_kernel<T, 8>;
        hipLaunchKernelGGL(kern, grid, dim3(kOrmThreads), 0, st, (int)n, (int)nc, R, ldr, strideR, B + c0 * ldb, ldb,
                           strideB, batch);
        const int rc = launch_check("trsm_regs_kernel");
        if (rc != GPUTILS_OK) return rc;
    }
    return GPUTILS_OK;
}

#define GPUTILS_QRR(T)                                                                                              \
    template int geqrf<T>(int64_t, int64_t, T *, int64_t, int64_t, T *, int64_t, int *, int64_t, hipStream_t);      \
    template int gels<T>(int64_t, int64_t, int64_t, T *, int64_t, int64_t, T *, int64_t, int64_t, int *, int64_t,   \
                         hipStream_t);                                                                              \
    template int trsm_upper<T>(int64_t, int64_t, const T *, int64_t, int64_t, T *, int64_t, int64_t, int64_t,       \
                               hipStream_t);                                                                        \
    template int ormqr<T>(int, int64_t, int64_t, int64_t, int64_t, const T *, int64_t, int64_t, const T *, int64_t, \
                          T *, int64_t, int64_t, int64_t, hipStream_t);
GPUTILS_QRR(float)
GPUTILS_QRR(double)

}  // namespace qrr
}  // namespace gputils
