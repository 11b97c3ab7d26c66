// trsm.hip -- triangular solve with many right-hand sides (DTRSM/STRSM) on
// gfx950, all 16 side/uplo/trans/diag forms.
//
// Replaces the vendor call at blas_level3/trsm.cc:52-72 (cublasDtrsm).
//
// Recursive blocking: the triangle is split in two halves (rounded to 64
// rows); one half is solved recursively, the off-diagonal block is applied to
// the other half's right-hand sides with the MFMA GEMM of gemm.hip (alpha = -1,
// beta = the solve's alpha), then the second half is solved.  Orders of at most
// 512 are solved in one launch, 16 right-hand sides per workgroup, on the FP64
// matrix cores (trsm_panel.hpp), the right side as the left side of the
// transposed system.
#include "trsm_panel.hpp"
#include "gpublas_dev.h"

int gpublas_gemm_d(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha,
                   const double *A, int lda, const double *B, int ldb, double beta, double *C,
                   int ldc);
int gpublas_gemm_s(hipStream_t s, char ta, char tb, int m, int n, int k, float alpha,
                   const float *A, int lda, const float *B, int ldb, float beta, float *C, int ldc);

namespace {

constexpr int NB = 64;

inline int gemm_t(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha,
                  const double *A, int lda, const double *B, int ldb, double beta, double *C,
                  int ldc)
{
    return gpublas_gemm_d(s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}
inline int gemm_t(hipStream_t s, char ta, char tb, int m, int n, int k, float alpha,
                  const float *A, int lda, const float *B, int ldb, float beta, float *C, int ldc)
{
    return gpublas_gemm_s(s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

// Base solve of an order of at most 128 * SB, one workgroup per 16 right-hand
// sides (trsm_panel.hpp).  The smaller SB, the more workgroups share a CU (4, 2,
// 1: LDS) and the shorter the prologue.  Measured with 4096 right-hand sides,
// left, lower, FP64 (FP32): order 16 8.0 -> 4.6 us (7.6 -> 4.5), 128 16.4 -> 8.3
// (30.7 -> 8.0), 256 23.6 -> 14.5 (50.0 -> 14.0), 512 67.4 -> 35.8 in one launch
// instead of two solves and a product (115 -> 34.7); order 64 with 100000 right-
// hand sides 151 -> 53 us (103 -> 55).  With every diagonal block substituted, FP64:
// order 16 6.2 us, 128 22.6, 256 43.8, 512 92.
template <typename T, int SB, bool KC>
__global__ __launch_bounds__(TP_THREADS) void trsm_base(int order, int n, double alpha, const T *A,
                                                        long lda, int transN, int lower, int unit,
                                                        T *B, long sstride, long rstride)
{
    __shared__ PanelLds<SB> s;
    const int c0 = blockIdx.x * 16;
    trsm_panel<T, SB, KC>(panel_args<T>(A, lda, transN, lower, unit, B + c0 * rstride, sstride, rstride,
                                    order, min(16, n - c0), alpha),
                      s);
}

template <typename T>
__global__ void zero_kernel(int m, int n, T *B, long ldb)
{
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long total = (long)m * n;
    for (; idx < total; idx += (long)gridDim.x * blockDim.x) B[idx % m + (idx / m) * ldb] = T(0);
}

inline int split(int m)
{
    int h = (m / 2 + NB - 1) / NB * NB;
    if (h >= m) h = m - NB;
    return h;
}

template <typename T>
struct Solve {
    hipStream_t s;
    int left, effLower, transN, nounit;
    const T *A;
    int lda;
    T *B;
    int ldb;

    // Solve on the sub-problem whose triangle starts at a (order `t`), with
    // right-hand sides at b (m x n, m = t for left, n = t for right).
    int base(int m, int n, T alpha, const T *a, T *b)
    {
        // right side: op(T)^T X^T = alpha B^T, the triangle of op(T)^T is
        // op(T) read the other way and of the other shape
        const int lower = left ? effLower : !effLower, tn = left ? transN : !transN;
        const int nrhs = left ? n : m, order = left ? m : n;
        const long ss = left ? 1 : ldb, rs = left ? ldb : 1;
        const unsigned blocks = (unsigned)ceil_div(nrhs, 16);
        auto k = order <= 128   ? (tn ? trsm_base<T, 1, false> : trsm_base<T, 1, true>)
                 : order <= 256 ? (tn ? trsm_base<T, 2, false> : trsm_base<T, 2, true>)
                                : (tn ? trsm_base<T, 4, false> : trsm_base<T, 4, true>);
        PROF_BEGIN(s, sizeof(T) == 8 ? "dtrsm_base" : "strsm_base");
        hipLaunchKernelGGL(k, dim3(blocks), dim3(TP_THREADS), 0, s, order, nrhs, (double)alpha, a,
                           (long)lda, tn, lower, !nounit, b, ss, rs);
        PROF_END(s);
        return (int)hipGetLastError();
    }

    int rec(int m, int n, T alpha, const T *a, T *b)
    {
        int err;
        const int t = left ? m : n;
        if (t <= 512) return base(m, n, alpha, a, b);
        const int t1 = split(t), t2 = t - t1;
        const T *a11 = a, *a22 = a + t1 + (long)t1 * lda;
        const T *a21 = a + t1, *a12 = a + (long)t1 * lda;  // stored blocks
        const char N = 'N', Tt = 'T';
        if (left) {
            T *b1 = b, *b2 = b + t1;
            if (effLower) {
                // op(A) = [[T11,0],[T21,T22]], T21 = A21 (N) or A12^T (T)
                if ((err = rec(t1, n, alpha, a11, b1))) return err;
                if (transN) err = gemm_t(s, N, N, t2, n, t1, T(-1), a21, lda, b1, ldb, alpha, b2, ldb);
                else err = gemm_t(s, Tt, N, t2, n, t1, T(-1), a12, lda, b1, ldb, alpha, b2, ldb);
                if (err) return err;
                return rec(t2, n, T(1), a22, b2);
            }
            // op(A) = [[T11,T12],[0,T22]], T12 = A12 (N) or A21^T (T)
            if ((err = rec(t2, n, alpha, a22, b2))) return err;
            if (transN) err = gemm_t(s, N, N, t1, n, t2, T(-1), a12, lda, b2, ldb, alpha, b1, ldb);
            else err = gemm_t(s, Tt, N, t1, n, t2, T(-1), a21, lda, b2, ldb, alpha, b1, ldb);
            if (err) return err;
            return rec(t1, n, T(1), a11, b1);
        }
        T *b1 = b, *b2 = b + (long)t1 * ldb;
        if (effLower) {
            // X [[T11,0],[T21,T22]] = alpha [B1,B2]
            if ((err = rec(m, t2, alpha, a22, b2))) return err;
            if (transN) err = gemm_t(s, N, N, m, t1, t2, T(-1), b2, ldb, a21, lda, alpha, b1, ldb);
            else err = gemm_t(s, N, Tt, m, t1, t2, T(-1), b2, ldb, a12, lda, alpha, b1, ldb);
            if (err) return err;
            return rec(m, t1, T(1), a11, b1);
        }
        // X [[T11,T12],[0,T22]] = alpha [B1,B2]
        if ((err = rec(m, t1, alpha, a11, b1))) return err;
        if (transN) err = gemm_t(s, N, N, m, t2, t1, T(-1), b1, ldb, a12, lda, alpha, b2, ldb);
        else err = gemm_t(s, N, Tt, m, t2, t1, T(-1), b1, ldb, a21, lda, alpha, b2, ldb);
        if (err) return err;
        return rec(m, t2, T(1), a22, b2);
    }
};

inline bool up(char c) { return c == 'U' || c == 'u'; }
inline bool isN(char c) { return c == 'N' || c == 'n'; }
inline bool isL(char c) { return c == 'L' || c == 'l'; }

template <typename T>
int trsm_entry(void *stream, char side, char uplo, char transa, char diag, int m, int n, T alpha,
               const T *A, int lda, T *B, int ldb)
{
    hipStream_t s = pick_stream(stream);
    if (m <= 0 || n <= 0) return 0;
    if (alpha == T(0)) {
        long total = (long)m * n;
        int blocks = (int)((total + 255) / 256);
        if (blocks > 8192) blocks = 8192;
        hipLaunchKernelGGL(zero_kernel<T>, dim3(blocks), dim3(256), 0, s, m, n, B, (long)ldb);
        return (int)hipGetLastError();
    }
    Solve<T> sv;
    sv.s = s;
    sv.left = isL(side);
    sv.transN = isN(transa);
    sv.effLower = (!up(uplo)) == sv.transN;
    sv.nounit = isN(diag);
    sv.A = A;
    sv.lda = lda;
    sv.B = B;
    sv.ldb = ldb;
    return sv.rec(m, n, alpha, A, B);
}

}  // namespace

extern "C" {

int gpublas_dev_dtrsm(void *stream, char side, char uplo, char transa, char diag, int m, int n,
                      double alpha, const double *d_A, int lda, double *d_B, int ldb)
{
    return trsm_entry<double>(stream, side, uplo, transa, diag, m, n, alpha, d_A, lda, d_B, ldb);
}

int gpublas_dev_strsm(void *stream, char side, char uplo, char transa, char diag, int m, int n,
                      float alpha, const float *d_A, int lda, float *d_B, int ldb)
{
    return trsm_entry<float>(stream, side, uplo, transa, diag, m, n, alpha, d_A, lda, d_B, ldb);
}

}  // extern "C"
