// gemm.hip -- LDS-tiled MFMA kernels for the real Level-3 routines on gfx950:
// DGEMM/SGEMM (all trans forms), DSYRK/SSYRK (one triangle), DSYMM/SSYMM.
//
// Replaces the vendor calls at blas_level3/gemm.cc:62-82 (cublasDgemm),
// syrk.cc:57-75 (cublasDsyrk) and symm.cc:57-78 (cublasDsymm).
//
// Products at least 32 wide in both dimensions run on the fast tile (any
// alignment, ragged edges by moved-back tiles, a tile shape by cost); the generic
// tile (both in gemm_tile.hpp) serves the rest and symmetric operands:
//  * SYRK is the same product with B = A (transposed), restricted to tiles
//    on and below (above) the diagonal and masked to the triangle;
//  * SYMM reads the symmetric operand from its stored triangle: per k-tile
//    the loader picks the direct layout, the mirrored (transposed) layout,
//    or a per-element select for tiles that straddle the diagonal.
#include "gemm_tile.hpp"
#include <algorithm>
#include "gpublas_dev.h"

namespace {
template <typename T, int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(GemmArgs<T> g)
{
    constexpr int PAD = 128 / (int)sizeof(T);
    __shared__ T As[2][BK][BM + PAD];
    __shared__ T Bs[2][BK][BN + PAD];

    int tm, tn;
    if (g.tri == SYM_NONE) {
        tm = blockIdx.x % g.tiles_m;
        tn = blockIdx.x / g.tiles_m;
    } else {
        int hi, lo;
        tri_decode(blockIdx.x, hi, lo);
        if (g.tri == SYM_LOWER) { tm = hi; tn = lo; } else { tm = lo; tn = hi; }
    }
    gemm_tile<T, BM, BN, BK>(g, tm, tn, As, Bs);
}

// Tile of block b of a rectangular grid: down the rows, column by column.  Blocks
// go round the eight XCDs, each with an L2 of its own, one by one, so with fewer
// than eight row tiles beside more column tiles every XCD would read most of B.
// Then the tiles of a column stay on one XCD: block 8 i + x takes XCD x's i-th tile
// of columns x, x + 8, ...; what is left of the columns runs in the plain order
// (FP64 NN 128 x 4096 x 4096 106 -> 78 us, 64 x 4096 x 4096 61 -> 43, NT 100 x 10000 x
// 256 23.2 -> 16.6; FP32 NT 128 x 4096 x 4096 75 -> 49).
template <typename T>
__device__ __forceinline__ void tile_at(const GemmArgs<T> &g, unsigned b, int &tm, int &tn)
{
    const unsigned rows = g.tiles_m, dealt = g.dealt * rows;
    const bool in = b < dealt;
    const unsigned i = in ? b >> 3 : b - dealt, q = i / rows;
    tm = i - q * rows;
    tn = in ? 8 * q + (b & 7) : g.dealt + q;
}
template <typename T> void set_tiles(GemmArgs<T> &g, int tiles_m, int tiles_n)
{
    g.tiles_m = tiles_m;
    g.tiles_n = tiles_n;
    g.dealt = tiles_m < 8 && tiles_n > tiles_m ? tiles_n / 8 * 8 : 0;
}

// Fast kernel: every tile of a product at least a tile wide in both dimensions,
// access patterns compile-time constants (PA / PB), operands of any alignment
// (gemm_fast_tile, tile shape S, lane offsets Off).
template <typename T, int S, int PA, int PB, int TRI, typename Off>
__global__ __launch_bounds__(256, 2) void gemm_fast_kernel(GemmArgs<T> g)
{
    typedef FastShape<T, S> F;
    __shared__ __attribute__((aligned(16))) T As[2][F::BK][F::LDA];
    __shared__ __attribute__((aligned(16))) T Bs[2][F::BK][F::LDB];

    int tm, tn;
    if (TRI == SYM_NONE) {
        if constexpr (S == 128) {
            // always many tiles: the plain order (8192^3 15.86 ms, 15.93 through tile_at)
            tm = blockIdx.x % g.tiles_m;
            tn = blockIdx.x / g.tiles_m;
        } else {
            tile_at(g, blockIdx.x, tm, tn);
        }
    } else {
        int hi, lo;
        tri_decode(blockIdx.x, hi, lo);
        if (TRI == SYM_LOWER) { tm = hi; tn = lo; } else { tm = lo; tn = hi; }
    }
    gemm_fast_tile<T, F::BM, F::BN, F::BK, F::NST, PA, PB, TRI, Off>(g, tm, tn, As, Bs);
}

// Split-K for problems with too few tiles to fill the chip and a long k:
// block b is tile b % tiles (shape S) over k chunk b / tiles (kchunk deep, a
// multiple of 16; the last one what is left), written unscaled to P[chunk] (m x
// n, leading dimension m); splitk_fold_kernel then forms alpha * (sum of chunks
// in chunk order) + beta * C.  The decomposition depends on the shape and the
// card alone, so the bits repeat from call to call; a call that is recorded into a
// graph, or finds no scratch, is not split and sums k in one run.
template <typename T, int S, int PA, int PB, typename Off>
__global__ __launch_bounds__(256, 2) void gemm_fast_splitk_kernel(GemmArgs<T> g, int kchunk, T *P)
{
    typedef FastShape<T, S> F;
    __shared__ __attribute__((aligned(16))) T As[2][F::BK][F::LDA];
    __shared__ __attribute__((aligned(16))) T Bs[2][F::BK][F::LDB];
    const int tiles = g.tiles_m * g.tiles_n;
    const int t = (int)(blockIdx.x % (unsigned)tiles), kc = (int)(blockIdx.x / (unsigned)tiles);
    const long koff = (long)kc * kchunk;
    GemmArgs<T> h = g;
    // element (o, k) of an operand is p[o + k*ld] (outer) or p[k + o*ld]
    h.a.p += PA == PAT_OUTER ? koff * g.a.ld : koff;
    h.b.p += PB == PAT_OUTER ? koff * g.b.ld : koff;
    h.k = min(kchunk, g.k - (int)koff);
    h.alpha = T(1);
    h.beta = T(0);
    h.C = P + (long)kc * g.m * g.n;
    h.ldc = g.m;
    int tm, tn;
    tile_at(g, t, tm, tn);
    gemm_fast_tile<T, F::BM, F::BN, F::BK, F::NST, PA, PB, SYM_NONE, Off>(h, tm, tn, As, Bs);
}

template <typename T>
__global__ __launch_bounds__(256) void splitk_fold_kernel(int m, int n, int ks, const T *P, T alpha,
                                                          T beta, T *C, long ldc)
{
    const long mn = (long)m * n;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < mn; e += (long)gridDim.x * 256) {
        T sum = P[e];
        for (int c = 1; c < ks; ++c) sum += P[(long)c * mn + e];
        const long i = e % m, j = e / m;
        T *cp = C + i + j * ldc;
        const T v = alpha * sum;
        *cp = beta == T(0) ? v : v + beta * *cp;
    }
}

// Scale (or zero) a triangle or rectangle of C: the alpha == 0 / k == 0
// paths of the netlib routines (beta == 0 stores exact zeros).
template <typename T>
__global__ void scale_kernel(int m, int n, T beta, T *C, long ldc, int tri)
{
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long total = (long)m * n;
    for (; idx < total; idx += (long)gridDim.x * blockDim.x) {
        long i = idx % m, j = idx / m;
        if (tri == SYM_LOWER && i < j) continue;
        if (tri == SYM_UPPER && i > j) continue;
        T *c = C + i + j * ldc;
        *c = beta == T(0) ? T(0) : beta * *c;
    }
}

template <typename T>
int launch_scale(hipStream_t s, int m, int n, T beta, T *C, long ldc, int tri)
{
    if (m <= 0 || n <= 0) return 0;
    long total = (long)m * n;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 8192) blocks = 8192;
    PROF_BEGIN(s, "scale");
    hipLaunchKernelGGL(scale_kernel<T>, dim3(blocks), dim3(256), 0, s, m, n, beta, C, ldc, tri);
    PROF_END(s);
    return (int)hipGetLastError();
}

template <typename T> const char *kname(int shape);
template <> const char *kname<double>(int shape)
{
    return shape == 128  ? "dgemm_fast_128x64"
           : shape == 64 ? "dgemm_fast_64x64"
           : shape == 32 ? "dgemm_fast_32x32"
                         : "dgemm_edge_64x64";
}
template <> const char *kname<float>(int shape)
{
    return shape == 128  ? "sgemm_fast_128x128"
           : shape == 64 ? "sgemm_fast_64x64"
           : shape == 32 ? "sgemm_fast_32x32"
                         : "sgemm_edge_64x64";
}

template <typename T, int S, typename Off = unsigned>
void launch_fast(hipStream_t s, const GemmArgs<T> &g, unsigned blocks)
{
#define GB_FAST(PA_, PB_, TRI_)                                                                  \
    hipLaunchKernelGGL((gemm_fast_kernel<T, S, PA_, PB_, TRI_, Off>), dim3(blocks), dim3(256), 0, s, g)
    const int pa = g.a.form, pb = g.b.form;
    if (g.tri == SYM_NONE) {
        if (pa == PAT_OUTER && pb == PAT_KCONT) GB_FAST(PAT_OUTER, PAT_KCONT, SYM_NONE);      // NN
        else if (pa == PAT_OUTER) GB_FAST(PAT_OUTER, PAT_OUTER, SYM_NONE);                    // NT
        else if (pb == PAT_KCONT) GB_FAST(PAT_KCONT, PAT_KCONT, SYM_NONE);                    // TN
        else GB_FAST(PAT_KCONT, PAT_OUTER, SYM_NONE);                                         // TT
        return;
    }
    if constexpr (FastShape<T, S>::BM == FastShape<T, S>::BN) {  // triangular grids: square tiles
        if (g.tri == SYM_LOWER) {
            if (pa == PAT_OUTER) GB_FAST(PAT_OUTER, PAT_OUTER, SYM_LOWER);  // A*A^T
            else GB_FAST(PAT_KCONT, PAT_KCONT, SYM_LOWER);                  // A^T*A
        } else {
            if (pa == PAT_OUTER) GB_FAST(PAT_OUTER, PAT_OUTER, SYM_UPPER);
            else GB_FAST(PAT_KCONT, PAT_KCONT, SYM_UPPER);
        }
    }
#undef GB_FAST
}

// Compute units of the current device.
long device_cus()
{
    static const long n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0) {
            (void)hipGetLastError();
            cus = 256;
        }
        return (long)cus;
    }();
    return n;
}

// Tile shape of a product on the fast kernel, by the time the busiest CU takes:
// its number of tiles times a tile's area over the rate that the shape reaches
// with the chip full (TFLOP/s at 4096^3: FP64 57 / 68 / 69.5 for 32 x 32, 64 x 64
// and 128 x 64; FP32 88 / 130 / 138 for 32 x 32, 64 x 64 and 128 x 128).  A 32 x 32
// tile is bound by L2: where a column's 32 rows (`skewed`: an operand read along
// its columns whose leading dimension is no multiple of 128 bytes) lie across one
// more cache line, it reaches three quarters of that (3001 x 768 x 768 NN FP64: 95
// us against 77 with 64 x 64, but 73 where the leading dimensions are even).  The
// large shape also needs several tiles a CU (FP64 eight, FP32 two), below which
// the 64 x 64 one measured the same.  Both sides, 32 against 64: FP64 512^3 8.2 and
// 20.8 us, 768^3 24.5 and 30.3, 1024^3 41.2 and 39.2, 1536^2 x 1024 84 and 98, 2047 x
// 1531 x 1789 209 and 173; FP32 512^3 6.0 and 11.9, 768^3 16.9 and 16.7, 1024^3 28.9
// and 21.9.  64 against 128: FP64 8192^2 x 2048 4.08 and 3.97 ms, FP32 2900^2 x 1500
// 229 and 287 us, 4096^3 1007 and 996.  0: narrower than every tile.
template <typename T>
double shape_cost(long m, long n, int tri, int shape, bool skewed)
{
    const bool dp = sizeof(T) == 8;
    const long bm = shape, bn = shape == 128 && dp ? 64 : shape, cus = device_cus();
    const long tm = (m + bm - 1) / bm, tn = (n + bn - 1) / bn;
    const long tiles = tri ? tm * (tm + 1) / 2 : tm * tn;
    const double rate = shape == 32   ? (dp ? 57 : 88) * (skewed ? 0.75 : 1)
                        : shape == 64 ? (dp ? 68 : 130)
                                      : (dp ? 69.5 : 138);
    return (double)((tiles + cus - 1) / cus * bm * bn) / rate;
}

template <typename T>
int fast_shape(long m, long n, int tri, bool skewed)
{
    const bool dp = sizeof(T) == 8;
    const long bn = dp ? 64 : 128;
    if (m < 32 || n < 32) return 0;
    int best = 32;
    double least = shape_cost<T>(m, n, tri, 32, skewed);
    if (m >= 64 && n >= 64) {
        const double c = shape_cost<T>(m, n, tri, 64, skewed);
        if (c <= least) best = 64, least = c;
    }
    if (m >= 128 && n >= bn && !(dp && tri) &&
        ((m + 127) / 128) * ((n + bn - 1) / bn) >= (dp ? 8 : 2) * device_cus() &&
        shape_cost<T>(m, n, tri, 128, skewed) <= least)
        best = 128;
    return best;
}

// An operand read along its columns whose columns start at any byte of a cache line.
template <typename T> bool skewed(const Operand<T> &o)
{
    return o.form == PAT_OUTER && (o.ld * sizeof(T)) % 128 != 0;
}

// Split-K launch of a rectangular product on S x S tiles, k cut into chunks of
// kchunk (a multiple of 16).  Returns -1 when no scratch is left, or while s records
// a graph (whose scratch would be held as long as the graph is), so the caller takes
// the ordinary grid.
template <typename T, int S, typename Off>
int launch_splitk(hipStream_t s, const GemmArgs<T> &g, int m, int n, int k, int kchunk)
{
    const int ks = ceil_div(k, kchunk);
    if (call_is_recorded()) return -1;
    T *P = (T *)dev_block((size_t)ks * m * n * sizeof(T));
    if (!P) return -1;
    GemmArgs<T> f = g;
    set_tiles(f, ceil_div(m, S), ceil_div(n, S));
    const unsigned blocks = (unsigned)((long)f.tiles_m * f.tiles_n * ks);
#define GB_SK(PA_, PB_)                                                                          \
    hipLaunchKernelGGL((gemm_fast_splitk_kernel<T, S, PA_, PB_, Off>), dim3(blocks), dim3(256), 0, s, \
                       f, kchunk, P)
    const int pa = g.a.form, pb = g.b.form;
    PROF_BEGIN(s, sizeof(T) == 8 ? "dgemm_splitk" : "sgemm_splitk");
    if (pa == PAT_OUTER && pb == PAT_KCONT) GB_SK(PAT_OUTER, PAT_KCONT);
    else if (pa == PAT_OUTER) GB_SK(PAT_OUTER, PAT_OUTER);
    else if (pb == PAT_KCONT) GB_SK(PAT_KCONT, PAT_KCONT);
    else GB_SK(PAT_KCONT, PAT_OUTER);
#undef GB_SK
    const long mn = (long)m * n;
    const unsigned fb = (unsigned)std::min<long>((mn + 255) / 256, 4096);
    hipLaunchKernelGGL(splitk_fold_kernel<T>, dim3(fb), dim3(256), 0, s, m, n, ks, (const T *)P,
                       g.alpha, g.beta, g.C, g.ldc);
    PROF_END(s);
    dev_release_after(P, s);
    return (int)hipGetLastError();
}

// How a rectangular product of at least 32 x 32 is split along k, if it is: shape 32
// where 32 x 32 tiles leave half of the CUs idle, as many chunks as fill them (at most
// 16, each at least 256 deep; the fold costs about 5 us, 256 of k about 3).  Else
// shape 64, two workgroups a CU, where that beats the unsplit `shape` by the cost rule
// above, the fold counted as 5 us and the partial sums' traffic at 3 TB/s: only a long
// k pays it.  (A skewed operand costs little where the chip is not full; FP32 tiles of
// 32 x 32 reach 100, 87 and 74 TFLOP/s with none, one and both operands contiguous
// along k.)  Unsplit and split: FP32 TN 512 x 512 x 16384 129 and 77 us, x 8192 66 and
// 45, 640 x 640 x 16384 232 and 117; FP64 NN 512 x 512 x 16384 159 and 142, 640 x 640 x
// 16384 275 and 220.
struct SplitPlan {
    int shape, kchunk;
};
template <typename T>
SplitPlan split_plan(long m, long n, long k, int shape, int along_k)
{
    if (k < 512) return {0, 0};
    const long cus = device_cus();
    auto chunk = [&](long tiles, long slots) {
        const long want = std::min(std::min(slots / tiles, 16l), k / 256);
        return want < 2 ? (int)k : ceil_div(ceil_div(k, want), 16) * 16;
    };
    const int c32 = chunk((long)ceil_div(m, 32) * ceil_div(n, 32), cus);
    if (c32 < k) return {32, c32};
    if (m < 64 || n < 64) return {0, 0};
    const long tiles = (long)ceil_div(m, 64) * ceil_div(n, 64);
    const int c64 = chunk(tiles, 2 * cus);
    if (c64 >= k) return {0, 0};
    const long ks = ceil_div(k, c64);
    const double us = 2e-6 * cus;  // of a unit of cost, per k
    const double one = shape_cost<T>(64, 64 * tiles * ks, SYM_NONE, 64, false) * c64 * us;
    const double fold = 5 + 2.0 * ks * m * n * sizeof(T) / 3e6;
    double whole = shape_cost<T>(m, n, SYM_NONE, shape, false) * k * us;
    if (sizeof(T) == 4 && shape == 32) whole *= 88.0 / (along_k == 0 ? 100 : along_k == 1 ? 87 : 74);
    if (one + fold >= whole) return {0, 0};
    return {64, c64};
}

// Core launcher: C = alpha*op(A)*op(B) + beta*C on an (optionally
// triangular) tile grid.  k > 0, alpha != 0 assumed.  Products at least 32 wide
// in both dimensions go to the fast kernel; the generic kernel takes the narrow
// ones and symmetric operands.  Leading dimensions past FAST_LD_MAX (`wide`) take its
// 64 x 64 and split-K forms with 64-bit offsets (FP64, leading dimension 2 x 10^7: 64 x
// 64 x 2048 TN 176 us on the generic kernel, 12 here; 2 x 10^7 rows of 64 columns times
// 64 x 64 5.8 and 4.5 ms).
template <typename T>
int launch_gemm(hipStream_t s, int m, int n, int k, T alpha, const Operand<T> &a,
                const Operand<T> &b, T beta, T *C, long ldc, int tri)
{
    GemmArgs<T> g;
    g.m = m; g.n = n; g.k = k;
    g.alpha = alpha; g.beta = beta;
    g.a = a; g.b = b;
    g.C = C; g.ldc = ldc;
    g.tri = tri;
    const bool wide = a.ld > FAST_LD_MAX || b.ld > FAST_LD_MAX;
    int shape = a.sym == SYM_NONE && b.sym == SYM_NONE
                    ? fast_shape<T>(m, n, tri, skewed(a) || skewed(b)) : 0;
    if (shape && tri == SYM_NONE) {
        const SplitPlan p = split_plan<T>(m, n, k, shape, (a.form == PAT_KCONT) + (b.form == PAT_KCONT));
        const int err = p.shape == 32 ? wide ? launch_splitk<T, 32, size_t>(s, g, m, n, k, p.kchunk)
                                             : launch_splitk<T, 32, unsigned>(s, g, m, n, k, p.kchunk)
                        : p.shape == 64 && !wide ? launch_splitk<T, 64, unsigned>(s, g, m, n, k, p.kchunk)
                                                 : -1;
        if (err >= 0) return err;
    }
    if (wide && shape) shape = m >= 64 && n >= 64 ? 64 : 0;
    const int bm = shape ? shape : 64, bn = shape == 128 && sizeof(T) == 8 ? 64 : bm;
    set_tiles(g, ceil_div(m, bm), ceil_div(n, bn));
    const long blocks = tri ? (long)g.tiles_m * (g.tiles_m + 1) / 2 : (long)g.tiles_m * g.tiles_n;
    PROF_BEGIN(s, kname<T>(shape));
    if (shape && wide) launch_fast<T, 64, size_t>(s, g, (unsigned)blocks);
    else if (shape == 128) launch_fast<T, 128>(s, g, (unsigned)blocks);
    else if (shape == 64) launch_fast<T, 64>(s, g, (unsigned)blocks);
    else if (shape == 32) launch_fast<T, 32>(s, g, (unsigned)blocks);
    else
        hipLaunchKernelGGL((gemm_mfma_kernel<T, 64, 64, 16>), dim3((unsigned)blocks), dim3(256), 0, s,
                           g);
    PROF_END(s);
    return (int)hipGetLastError();
}

template <typename T>
int gemm_entry(void *stream, char transa, char transb, int m, int n, int k, T alpha, const T *A,
               int lda, const T *B, int ldb, T beta, T *C, int ldc)
{
    hipStream_t s = pick_stream(stream);
    if (m <= 0 || n <= 0) return 0;
    if (alpha == T(0) || k <= 0) {
        if (beta == T(1)) return 0;
        return launch_scale<T>(s, m, n, beta, C, ldc, SYM_NONE);
    }
    Operand<T> a = make_op<T>(A, lda, m, is_n(transa) ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    Operand<T> b = make_op<T>(B, ldb, n, is_n(transb) ? PAT_KCONT : PAT_OUTER, SYM_NONE);
    return launch_gemm<T>(s, m, n, k, alpha, a, b, beta, C, ldc, SYM_NONE);
}

template <typename T>
int syrk_entry(void *stream, char uplo, char trans, int n, int k, T alpha, const T *A, int lda,
               T beta, T *C, int ldc)
{
    hipStream_t s = pick_stream(stream);
    const int tri = is_u(uplo) ? SYM_UPPER : SYM_LOWER;
    if (n <= 0) return 0;
    if (alpha == T(0) || k <= 0) {
        if (beta == T(1)) return 0;
        return launch_scale<T>(s, n, n, beta, C, ldc, tri);
    }
    // trans N: C = A*A^T  -> op(A) = A (n x k), op(B) = A^T
    // trans T: C = A^T*A  -> op(A) = A^T,       op(B) = A
    const bool nt = is_n(trans);
    Operand<T> a = make_op<T>(A, lda, n, nt ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    Operand<T> b = make_op<T>(A, lda, n, nt ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    return launch_gemm<T>(s, n, n, k, alpha, a, b, beta, C, ldc, tri);
}

// Full symmetric matrix S (n x n, leading dimension lds) from the stored
// triangle of A: one workgroup per 64 x 64 tile of S.  Tiles inside the
// stored triangle are copied, tiles in the other one are the transposed
// mirror tile (through LDS, so both sides stay coalesced), diagonal tiles
// pick per element.  Every thread issues its 16 loads before its stores.
template <typename T>
__global__ __launch_bounds__(256) void symmetrize_kernel(int n, const T *__restrict__ A, long lda,
                                                         int lower, T *__restrict__ S, long lds)
{
    __shared__ T t[64][65];
    const int I = blockIdx.x, J = blockIdx.y;
    const int i0 = I * 64, j0 = J * 64;
    const bool diag = I == J, direct = lower ? I > J : I < J;
    // source tile: (I, J) itself, or its mirror (J, I); element (a, b) of it
    // is A[(r0 + a) + (c0 + b) * lda]
    const int r0 = direct || diag ? i0 : j0, c0 = direct || diag ? j0 : i0;
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int idx = threadIdx.x + 256 * u, a = idx & 63, b = idx >> 6;
        v[u] = (r0 + a < n && c0 + b < n) ? A[(r0 + a) + (long)(c0 + b) * lda] : T(0);
    }
    if (direct) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int idx = threadIdx.x + 256 * u, a = idx & 63, b = idx >> 6;
            if (i0 + a < n && j0 + b < n) S[(i0 + a) + (long)(j0 + b) * lds] = v[u];
        }
        return;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int idx = threadIdx.x + 256 * u;
        t[idx & 63][idx >> 6] = v[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int idx = threadIdx.x + 256 * u, a = idx & 63, b = idx >> 6;
        if (i0 + a >= n || j0 + b >= n) continue;
        // S(i0+a, j0+b): mirror tile -> A(j0+b, i0+a) = t[b][a]; diagonal
        // tile -> the stored one of (a, b) and (b, a)
        const bool stored = lower ? a >= b : a <= b;
        S[(i0 + a) + (long)(j0 + b) * lds] = (diag && stored) ? t[a][b] : t[b][a];
    }
}

// C = alpha*op(A)*op(B) where one factor is a triangle: tile
// (tm, tn) runs only over the k range where that factor is nonzero (the
// other products are exact zeros), so a triangular multiply costs half a
// GEMM.  KR: 1 k < (tm+1)*BM, 2 k >= tm*BM (left factor lower / upper),
// 3 k >= tn*BN, 4 k < (tn+1)*BN (right factor lower / upper).  Operand
// pointers are shifted to the range start as in the split-K kernel; tiles
// are dispatched longest range first.  (A ragged last tile is moved back, but
// stores only its own rows and columns, for which the range is right.)
template <typename T, int S, int PA, int PB, int KR>
__global__ __launch_bounds__(256, 2) void gemm_fast_krange_kernel(GemmArgs<T> g)
{
    typedef FastShape<T, S> F;
    constexpr int BM = F::BM, BN = F::BN;
    __shared__ __attribute__((aligned(16))) T As[2][F::BK][F::LDA];
    __shared__ __attribute__((aligned(16))) T Bs[2][F::BK][F::LDB];
    // longest ranges first, so the last round holds the shortest tiles
    const int b = (int)blockIdx.x;
    int tm, tn;
    if (KR == 1 || KR == 2) {
        tm = b / g.tiles_n;
        if (KR == 1) tm = g.tiles_m - 1 - tm;
        tn = b % g.tiles_n;
    } else {
        tn = b / g.tiles_m;
        if (KR == 4) tn = g.tiles_n - 1 - tn;
        tm = b % g.tiles_m;
    }
    int kb = 0, ke = g.k;
    if (KR == 1) ke = min(g.k, (tm + 1) * BM);
    if (KR == 2) kb = tm * BM;
    if (KR == 3) kb = tn * BN;
    if (KR == 4) ke = min(g.k, (tn + 1) * BN);
    GemmArgs<T> h = g;
    h.a.p += PA == PAT_OUTER ? (long)kb * g.a.ld : kb;
    h.b.p += PB == PAT_OUTER ? (long)kb * g.b.ld : kb;
    h.k = ke - kb;
    gemm_fast_tile<T, BM, BN, F::BK, F::NST, PA, PB, SYM_NONE>(h, tm, tn, As, Bs);
}

// Full n x n matrix of a triangle of A: the stored triangle copied, zeros
// elsewhere, ones on the diagonal when `unit` (the diagonal of A is then not
// read).  One workgroup per 64 x 64 tile; coalesced on both sides.
template <typename T>
__global__ __launch_bounds__(256) void triangle_kernel(int n, const T *__restrict__ A, long lda,
                                                       int lower, int unit, T *__restrict__ Tm,
                                                       long ldt)
{
    const int i0 = blockIdx.x * 64, j0 = blockIdx.y * 64;
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int idx = threadIdx.x + 256 * u, i = i0 + (idx & 63), j = j0 + (idx >> 6);
        const bool in = i < n && j < n && (lower ? i >= j : i <= j) && !(unit && i == j);
        v[u] = in ? A[i + (long)j * lda] : (unit && i == j ? T(1) : T(0));
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int idx = threadIdx.x + 256 * u, i = i0 + (idx & 63), j = j0 + (idx >> 6);
        if (i < n && j < n) Tm[i + (long)j * ldt] = v[u];
    }
}

template <typename T>
int symm_entry(void *stream, char side, char uplo, int m, int n, T alpha, const T *A, int lda,
               const T *B, int ldb, T beta, T *C, int ldc)
{
    hipStream_t s = pick_stream(stream);
    if (m <= 0 || n <= 0) return 0;
    if (alpha == T(0)) {
        if (beta == T(1)) return 0;
        return launch_scale<T>(s, m, n, beta, C, ldc, SYM_NONE);
    }
    const int sym = is_u(uplo) ? SYM_UPPER : SYM_LOWER;
    // From order 256 up, the stored triangle is first expanded into a full
    // symmetric matrix (one pass over na^2 elements) so the product runs on
    // the fast GEMM kernels; the same products in the same k order (but where k
    // is split).
    const int na = is_l(side) ? m : n;
    if (na >= 256) {
        const long lds = (na + 7) / 8 * 8;
        T *S = (T *)dev_block((size_t)lds * na * sizeof(T));
        if (S) {
            const unsigned tiles = (unsigned)ceil_div(na, 64);
            PROF_BEGIN(s, "symmetrize");
            hipLaunchKernelGGL(symmetrize_kernel<T>, dim3(tiles, tiles), dim3(256), 0, s, na, A,
                               (long)lda, sym == SYM_LOWER ? 1 : 0, S, lds);
            PROF_END(s);
            int err = (int)hipGetLastError();
            if (!err) {
                if (is_l(side))
                    err = launch_gemm<T>(s, m, n, m, alpha,
                                         make_op<T>(S, lds, m, PAT_OUTER, SYM_NONE),
                                         make_op<T>(B, ldb, n, PAT_KCONT, SYM_NONE), beta, C, ldc,
                                         SYM_NONE);
                else
                    err = launch_gemm<T>(s, m, n, n, alpha,
                                         make_op<T>(B, ldb, m, PAT_OUTER, SYM_NONE),
                                         make_op<T>(S, lds, n, PAT_KCONT, SYM_NONE), beta, C, ldc,
                                         SYM_NONE);
            }
            dev_release_after(S, s);
            return err;
        }
    }
    if (is_l(side)) {
        // C = alpha*A*B + beta*C, A symmetric m x m: k = m
        Operand<T> a = make_op<T>(A, lda, m, PAT_OUTER, sym);
        Operand<T> b = make_op<T>(B, ldb, n, PAT_KCONT, SYM_NONE);
        return launch_gemm<T>(s, m, n, m, alpha, a, b, beta, C, ldc, SYM_NONE);
    }
    // C = alpha*B*A + beta*C, A symmetric n x n: k = n
    Operand<T> a = make_op<T>(B, ldb, m, PAT_OUTER, SYM_NONE);
    Operand<T> b = make_op<T>(A, lda, n, PAT_KCONT, sym);
    return launch_gemm<T>(s, m, n, n, alpha, a, b, beta, C, ldc, SYM_NONE);
}

// Triangular-k product (see gemm_fast_krange_kernel); -1 when the shape or
// the operands do not allow the fast tiles (the caller then runs the
// ordinary full-k GEMM).  beta = 0.
template <typename T, int S>
int launch_krange(hipStream_t s, int m, int n, int k, T alpha, const Operand<T> &a,
                  const Operand<T> &b, T *C, long ldc, int kr)
{
    constexpr int BM = FastShape<T, S>::BM, BN = FastShape<T, S>::BN;
    if (m < BM || n < BN || a.ld > FAST_LD_MAX || b.ld > FAST_LD_MAX) return -1;
    GemmArgs<T> g;
    g.m = m; g.n = n; g.k = k;
    g.alpha = alpha; g.beta = T(0);
    g.a = a; g.b = b;
    g.C = C; g.ldc = ldc;
    g.tri = SYM_NONE;
    set_tiles(g, ceil_div(m, BM), ceil_div(n, BN));
    const unsigned blocks = (unsigned)(g.tiles_m * g.tiles_n);
#define GB_KR(PA_, PB_)                                                                          \
    do {                                                                                         \
        if (kr == 1) hipLaunchKernelGGL((gemm_fast_krange_kernel<T, S, PA_, PB_, 1>), dim3(blocks), dim3(256), 0, s, g); \
        else if (kr == 2) hipLaunchKernelGGL((gemm_fast_krange_kernel<T, S, PA_, PB_, 2>), dim3(blocks), dim3(256), 0, s, g); \
        else if (kr == 3) hipLaunchKernelGGL((gemm_fast_krange_kernel<T, S, PA_, PB_, 3>), dim3(blocks), dim3(256), 0, s, g); \
        else hipLaunchKernelGGL((gemm_fast_krange_kernel<T, S, PA_, PB_, 4>), dim3(blocks), dim3(256), 0, s, g); \
    } while (0)
    const int pa = a.form, pb = b.form;
    PROF_BEGIN(s, sizeof(T) == 8 ? "dgemm_krange" : "sgemm_krange");
    if (pa == PAT_OUTER && pb == PAT_KCONT) GB_KR(PAT_OUTER, PAT_KCONT);
    else if (pa == PAT_OUTER) GB_KR(PAT_OUTER, PAT_OUTER);
    else if (pb == PAT_KCONT) GB_KR(PAT_KCONT, PAT_KCONT);
    else GB_KR(PAT_KCONT, PAT_OUTER);
#undef GB_KR
    PROF_END(s);
    return (int)hipGetLastError();
}

// C = alpha*op(A)*op(B)^T + alpha*op(B)*op(A)^T + beta*C on the uplo triangle
// (op(X) = X, n x k, for trans N; X^T for trans T): two triangular-grid
// products, the second accumulating onto the first.
template <typename T>
int syr2k_entry(void *stream, char uplo, char trans, int n, int k, T alpha, const T *A, int lda,
                const T *B, int ldb, T beta, T *C, int ldc)
{
    hipStream_t s = pick_stream(stream);
    const int tri = is_u(uplo) ? SYM_UPPER : SYM_LOWER;
    if (n <= 0) return 0;
    if (alpha == T(0) || k <= 0) {
        if (beta == T(1)) return 0;
        return launch_scale<T>(s, n, n, beta, C, ldc, tri);
    }
    const bool nt = is_n(trans);
    Operand<T> a = make_op<T>(A, lda, n, nt ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    Operand<T> b = make_op<T>(B, ldb, n, nt ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    int err = launch_gemm<T>(s, n, n, k, alpha, a, b, beta, C, ldc, tri);
    if (!err) err = launch_gemm<T>(s, n, n, k, alpha, b, a, T(1), C, ldc, tri);
    return err;
}

// B := alpha*op(A)*B (side L) or alpha*B*op(A) (side R), A triangular: the
// triangle is expanded into a full matrix (zeros outside it, ones on a unit
// diagonal), the product runs on the GEMM tiles into a workspace -- each tile
// only over the k range where the triangle is nonzero when the tiles are
// full -- and the workspace is copied over B.
template <typename T>
int trmm_entry(void *stream, char side, char uplo, char transa, char diag, int m, int n, T alpha,
               const T *A, int lda, T *B, int ldb)
{
    hipStream_t s = pick_stream(stream);
    if (m <= 0 || n <= 0) return 0;
    if (alpha == T(0)) return launch_scale<T>(s, m, n, T(0), B, ldb, SYM_NONE);
    const bool left = is_l(side);
    const int na = left ? m : n;
    const long ldt = (na + 7) / 8 * 8, ldw = (m + 7) / 8 * 8;
    T *Tm = (T *)dev_block((size_t)ldt * na * sizeof(T));
    T *W = (T *)dev_block((size_t)ldw * n * sizeof(T));
    if (!Tm || !W) {
        gpublas_dev_release(Tm);
        gpublas_dev_release(W);
        return (int)hipErrorOutOfMemory;
    }
    const unsigned tiles = (unsigned)ceil_div(na, 64);
    PROF_BEGIN(s, "triangle");
    hipLaunchKernelGGL(triangle_kernel<T>, dim3(tiles, tiles), dim3(256), 0, s, na, A, (long)lda,
                       is_u(uplo) ? 0 : 1, (diag == 'U' || diag == 'u') ? 1 : 0, Tm, ldt);
    PROF_END(s);
    int err = (int)hipGetLastError();
    const bool tn = is_n(transa);
    // op(A) lower: the transposed upper triangle, or the lower one as stored
    const bool oplower = is_u(uplo) ? !tn : tn;
    if (!err) {
        const Operand<T> a = left ? make_op<T>(Tm, ldt, m, tn ? PAT_OUTER : PAT_KCONT, SYM_NONE)
                                  : make_op<T>(B, ldb, m, PAT_OUTER, SYM_NONE);
        const Operand<T> b = left ? make_op<T>(B, ldb, n, PAT_KCONT, SYM_NONE)
                                  : make_op<T>(Tm, ldt, n, tn ? PAT_KCONT : PAT_OUTER, SYM_NONE);
        const int k = left ? m : n;
        const int kr = left ? (oplower ? 1 : 2) : (oplower ? 3 : 4);
        // the full product's shape; FP64 from 24 large tiles a CU on, as their ranges
        // even out late (8192^2 9.27 ms on 64 x 64 tiles, 8.42 on 128 x 64; 6144^2 3.44
        // and 3.56, 4096^2 1.07 and 1.11)
        const bool many = sizeof(T) == 4 ||
                          (long)ceil_div(m, 128) * ceil_div(n, 64) >= 24 * device_cus();
        err = many && fast_shape<T>(m, n, SYM_NONE, false) == 128
                  ? launch_krange<T, 128>(s, m, n, k, alpha, a, b, W, ldw, kr)
                  : launch_krange<T, 64>(s, m, n, k, alpha, a, b, W, ldw, kr);
        if (err < 0) err = launch_gemm<T>(s, m, n, k, alpha, a, b, T(0), W, ldw, SYM_NONE);
    }
    if (!err)
        err = (int)hipMemcpy2DAsync(B, (size_t)ldb * sizeof(T), W, (size_t)ldw * sizeof(T),
                                    (size_t)m * sizeof(T), (size_t)n, hipMemcpyDeviceToDevice, s);
    dev_release_after(Tm, s);
    dev_release_after(W, s);
    return err;
}

}  // namespace

// Shared with trsm.hip: plain GEMM on device pointers.
int gpublas_gemm_d(hipStream_t s, char ta, char tb, int m, int n, int k, double alpha,
                   const double *A, int lda, const double *B, int ldb, double beta, double *C,
                   int ldc)
{
    return gemm_entry<double>(s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}
int gpublas_gemm_s(hipStream_t s, char ta, char tb, int m, int n, int k, float alpha,
                   const float *A, int lda, const float *B, int ldb, float beta, float *C, int ldc)
{
    return gemm_entry<float>(s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

// Shared with cplx.hip: the uplo triangle of alpha op(A) op(B) + beta C on
// the triangular tile grid (op(A) n x k, op(B) k x n); the rest of C is not
// touched.
template <typename T>
int gemm_tri(hipStream_t s, char uplo, char ta, char tb, int n, int k, T alpha, const T *A,
             int lda, const T *B, int ldb, T beta, T *C, int ldc)
{
    const int tri = is_u(uplo) ? SYM_UPPER : SYM_LOWER;
    if (n <= 0) return 0;
    if (alpha == T(0) || k <= 0) {
        if (beta == T(1)) return 0;
        return launch_scale<T>(s, n, n, beta, C, ldc, tri);
    }
    Operand<T> a = make_op<T>(A, lda, n, is_n(ta) ? PAT_OUTER : PAT_KCONT, SYM_NONE);
    Operand<T> b = make_op<T>(B, ldb, n, is_n(tb) ? PAT_KCONT : PAT_OUTER, SYM_NONE);
    return launch_gemm<T>(s, n, n, k, alpha, a, b, beta, C, ldc, tri);
}
int gpublas_gemm_tri_d(hipStream_t s, char uplo, char ta, char tb, int n, int k, double alpha,
                       const double *A, int lda, const double *B, int ldb, double beta, double *C,
                       int ldc)
{
    return gemm_tri<double>(s, uplo, ta, tb, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}
int gpublas_gemm_tri_s(hipStream_t s, char uplo, char ta, char tb, int n, int k, float alpha,
                       const float *A, int lda, const float *B, int ldb, float beta, float *C,
                       int ldc)
{
    return gemm_tri<float>(s, uplo, ta, tb, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

extern "C" {

int gpublas_dev_dgemm(void *stream, char transa, char transb, int m, int n, int k, double alpha,
                      const double *d_A, int lda, const double *d_B, int ldb, double beta,
                      double *d_C, int ldc)
{
    return gemm_entry<double>(stream, transa, transb, m, n, k, alpha, d_A, lda, d_B, ldb, beta,
                              d_C, ldc);
}

int gpublas_dev_sgemm(void *stream, char transa, char transb, int m, int n, int k, float alpha,
                      const float *d_A, int lda, const float *d_B, int ldb, float beta,
                      float *d_C, int ldc)
{
    return gemm_entry<float>(stream, transa, transb, m, n, k, alpha, d_A, lda, d_B, ldb, beta,
                             d_C, ldc);
}

int gpublas_dev_dsyrk(void *stream, char uplo, char trans, int n, int k, double alpha,
                      const double *d_A, int lda, double beta, double *d_C, int ldc)
{
    return syrk_entry<double>(stream, uplo, trans, n, k, alpha, d_A, lda, beta, d_C, ldc);
}

int gpublas_dev_ssyrk(void *stream, char uplo, char trans, int n, int k, float alpha,
                      const float *d_A, int lda, float beta, float *d_C, int ldc)
{
    return syrk_entry<float>(stream, uplo, trans, n, k, alpha, d_A, lda, beta, d_C, ldc);
}

int gpublas_dev_dsyr2k(void *stream, char uplo, char trans, int n, int k, double alpha,
                       const double *d_A, int lda, const double *d_B, int ldb, double beta,
                       double *d_C, int ldc)
{
    return syr2k_entry<double>(stream, uplo, trans, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
}

int gpublas_dev_ssyr2k(void *stream, char uplo, char trans, int n, int k, float alpha,
                       const float *d_A, int lda, const float *d_B, int ldb, float beta,
                       float *d_C, int ldc)
{
    return syr2k_entry<float>(stream, uplo, trans, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
}

int gpublas_dev_dtrmm(void *stream, char side, char uplo, char transa, char diag, int m, int n,
                      double alpha, const double *d_A, int lda, double *d_B, int ldb)
{
    return trmm_entry<double>(stream, side, uplo, transa, diag, m, n, alpha, d_A, lda, d_B, ldb);
}

int gpublas_dev_strmm(void *stream, char side, char uplo, char transa, char diag, int m, int n,
                      float alpha, const float *d_A, int lda, float *d_B, int ldb)
{
    return trmm_entry<float>(stream, side, uplo, transa, diag, m, n, alpha, d_A, lda, d_B, ldb);
}

int gpublas_dev_dsymm(void *stream, char side, char uplo, int m, int n, double alpha,
                      const double *d_A, int lda, const double *d_B, int ldb, double beta,
                      double *d_C, int ldc)
{
    return symm_entry<double>(stream, side, uplo, m, n, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
}

int gpublas_dev_ssymm(void *stream, char side, char uplo, int m, int n, float alpha,
                      const float *d_A, int lda, const float *d_B, int ldb, float beta,
                      float *d_C, int ldc)
{
    return symm_entry<float>(stream, side, uplo, m, n, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
}

}  // extern "C"
