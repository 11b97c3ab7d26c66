// gemm_tile.hpp -- the generic LDS-tiled MFMA GEMM tile shared by the
// per-call kernels (gemm.hip) and the grouped persistent kernels of the
// serving loop (group.hip).  Every form of the tile (generic, fast, guarded)
// sums k in the same order, so neither the shape of a tile nor the path changes a
// product's bits; a split of k does, and the two paths have a rule each for it.
//
// Tile scheme:
//  * a 256-thread workgroup owns a BM x BN tile of C; its 4 waves split the
//    tile 2 x 2 and each wave accumulates (BM/2) x (BN/2) with
//    v_mfma_f64_16x16x4_f64 (FP64) or v_mfma_f32_16x16x4_f32 (FP32);
//  * op(A) and op(B) tiles of depth BK stream through double-buffered LDS,
//    stored k-major ([BK][BM+PAD]) so each MFMA operand fragment is one
//    ds_read per lane; the next k-tile's global loads are in flight while
//    the current one is multiplied;
//  * the MFMA is issued with the B fragment first, so the accumulator holds
//    C^T and 16 consecutive lanes own 16 consecutive rows of one column of
//    C: the epilogue reads/writes C in 128-byte column segments;
//  * the k index advances in steps of 4 in increasing order whatever BM, BN
//    and BK are, so every tile shape gives the same result bits.
#pragma once
#include "devcommon.hpp"
#include <math.h>

namespace {

enum { PAT_OUTER = 0, PAT_KCONT = 1, PAT_ELEM = 2 };
enum { SYM_NONE = 0, SYM_LOWER = 1, SYM_UPPER = 2 };

// One operand of the product as the loader sees it: element (o, k) of the
// operand tile, where o is the row of op(A) (or the column of op(B)) and k
// the reduction index.  `form` says which of the two address forms is the
// natural one: OUTER -> p[o + k*ld], KCONT -> p[k + o*ld].  For a symmetric
// operand (sym != 0) the stored matrix S is addressed S[r + c*ld] with
// (r, c) = (o, k) for OUTER and (k, o) for KCONT, and only the `sym`
// triangle of S may be read.
template <typename T>
struct Operand {
    const T *p;
    long ld;
    int olim;   // rows of op(A) / columns of op(B)
    int form;   // PAT_OUTER or PAT_KCONT
    int sym;    // SYM_*
    int vec_ok; // p 16-B aligned and ld a multiple of the vector width
};

template <typename T>
struct GemmArgs {
    int m, n, k;
    T alpha, beta;
    Operand<T> a, b;
    T *C;
    long ldc;
    int tiles_m, tiles_n;
    int dealt;  // columns of tiles dealt to the XCDs one by one (tile_at)
    int tri;  // 0 rectangular grid, SYM_LOWER / SYM_UPPER: triangular tile grid + mask
};

__device__ __forceinline__ bool stored(int sym, long r, long c)
{
    return sym == SYM_LOWER ? r >= c : r <= c;
}

// Pattern for the tile o in [o0, o0+R), k in [k0, k0+BK).
// LDS tile layout: element (k, o) of a staged tile lives at column
// o ^ lds_swz<T, R>(k).  Rows are BM + 128 bytes apart (0 modulo the 64 banks
// for every other row), so the transposed stores of a k-contiguous operand
// would put the 8 (double) or 4 (float) k rows one wave writes for a
// column on the same banks; the XOR moves each row pair (quad) to its own
// bank group.  It keeps 16-byte vectors and 32-column blocks intact, so
// vector stores and the MFMA fragment reads stay conflict-free.
// (R: columns of the tile, within which the XOR has to stay.)
template <typename T, int R> __device__ __forceinline__ int lds_swz(int k)
{
    return (sizeof(T) == 8 ? 4 * (k >> 1) : 16 * (k >> 2)) & (R - 1);
}

template <typename T, int R, int BK>
__device__ __forceinline__ int tile_pattern(const Operand<T> &op, int o0, int k0, int K)
{
    const bool full = (o0 + R <= op.olim) && (k0 + BK <= K);
    if (op.sym == SYM_NONE) return (full && op.vec_ok) ? op.form : PAT_ELEM;
    if (!full || !op.vec_ok) return PAT_ELEM;
    // (r, c) ranges of the tile in the stored matrix
    long rlo, rhi, clo, chi;
    if (op.form == PAT_OUTER) { rlo = o0; rhi = o0 + R - 1; clo = k0; chi = k0 + BK - 1; }
    else { rlo = k0; rhi = k0 + BK - 1; clo = o0; chi = o0 + R - 1; }
    bool all_direct, all_mirror;
    if (op.sym == SYM_LOWER) { all_direct = rlo >= chi; all_mirror = rhi <= clo; }
    else { all_direct = rhi <= clo; all_mirror = rlo >= chi; }
    if (all_direct) return op.form;
    if (all_mirror) return op.form == PAT_OUTER ? PAT_KCONT : PAT_OUTER;
    return PAT_ELEM;
}

template <typename T>
__device__ __forceinline__ T elem_load(const Operand<T> &op, long o, long k, int K)
{
    if (o >= op.olim || k >= K) return T(0);
    long r = op.form == PAT_OUTER ? o : k;
    long c = op.form == PAT_OUTER ? k : o;
    if (op.sym != SYM_NONE && !stored(op.sym, r, c)) { long t = r; r = c; c = t; }
    return op.p[r + c * op.ld];
}

// Global -> registers.  Each thread owns NV vectors of VEC elements.  For
// PAT_OUTER and PAT_ELEM the vector runs along o; for PAT_KCONT along k.
template <typename T, int R, int BK>
struct TileLoader {
    static constexpr int VEC = 16 / (int)sizeof(T);
    static constexpr int NV = R * BK / VEC / 256;
    static_assert(NV >= 1, "tile too small for 256 threads");
    static_assert((R & (R - 1)) == 0, "lds_swz must stay inside the tile rows");
    typedef T Vec __attribute__((ext_vector_type(VEC)));

    __device__ __forceinline__ static void load(const Operand<T> &op, int o0, int k0, int K,
                                                int pat, Vec (&st)[NV])
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int v = t + r * 256;
            if (pat == PAT_OUTER) {
                const int o = (v % (R / VEC)) * VEC, kk = v / (R / VEC);
                st[r] = *(const Vec *)(op.p + (long)(o0 + o) + (long)(k0 + kk) * op.ld);
            } else if (pat == PAT_KCONT) {
                const int kk = (v % (BK / VEC)) * VEC, o = v / (BK / VEC);
                st[r] = *(const Vec *)(op.p + (long)(k0 + kk) + (long)(o0 + o) * op.ld);
            } else {
                const int o = (v % (R / VEC)) * VEC, kk = v / (R / VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) st[r][e] = elem_load(op, o0 + o + e, k0 + kk, K);
            }
        }
    }

    // Fast path: the R rows of the tile all exist, pattern fixed at compile
    // time.  `base` is the tile's first element (uniform over the workgroup),
    // so a load is one 32-bit lane offset (voff) on a scalar address that the
    // scalar unit advances; per-lane 64-bit addresses for the 2 * NV loads of
    // a k-tile cost the registers that the fragment double buffer needs.  (Off:
    // unsigned up to FAST_LD_MAX, size_t past it.)
    // Operands may have any alignment: 16-byte loads that are only
    // element-aligned are legal in global memory.
    typedef T VecU __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
    static constexpr int OUTER_K = 256 * VEC / R;   // k rows one pass covers (PAT_OUTER)
    static constexpr int KCONT_O = 256 * VEC / BK;  // operand rows one pass covers (PAT_KCONT)

    template <int PAT, typename Off> __device__ __forceinline__ static Off voff(long ld)
    {
        const unsigned t = threadIdx.x;
        const Off l = (Off)ld;
        return (PAT == PAT_OUTER ? (t % (R / VEC)) * VEC + (t / (R / VEC)) * l
                                 : (t % (BK / VEC)) * VEC + (t / (BK / VEC)) * l) *
               (Off)sizeof(T);
    }
    template <int PAT, typename Off>
    __device__ __forceinline__ static void load_pat(const T *base, long ld, Off vo, Vec (&st)[NV])
    {
        const long step = (PAT == PAT_OUTER ? OUTER_K : KCONT_O) * ld;
#pragma unroll
        for (int r = 0; r < NV; ++r)
            st[r] = *(const VecU *)((const char *)(base + r * step) + (size_t)vo);
    }
    // The last k-tile when only krem < BK of its k rows exist: rows past them
    // read as zero (their addresses stay on the last row that exists).
    template <int PAT, typename Off>
    __device__ __forceinline__ static void load_ktail(const T *base, long ld, int krem,
                                                      Vec (&st)[NV])
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            if (PAT == PAT_OUTER) {
                const int o = (t % (R / VEC)) * VEC, kk = t / (R / VEC) + r * OUTER_K;
                const Off off = (Off)min(kk, krem - 1) * (Off)ld + (Off)o;
                const Vec x = *(const VecU *)((const char *)base + (size_t)(off * (Off)sizeof(T)));
#pragma unroll
                for (int e = 0; e < VEC; ++e) st[r][e] = kk < krem ? x[e] : T(0);
            } else {
                const int kk = (t % (BK / VEC)) * VEC, o = t / (BK / VEC);
                const T *row = base + r * (KCONT_O * ld);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const Off off = (Off)o * (Off)ld + (Off)min(kk + e, krem - 1);
                    const T x = *(const T *)((const char *)row + (size_t)(off * (Off)sizeof(T)));
                    st[r][e] = kk + e < krem ? x : T(0);
                }
            }
        }
    }

    // A ragged tile with the pattern fixed at compile time: element loads,
    // zero outside the operand (o >= olim or k >= K; the address is clamped
    // to the operand's first element there, so no load is skipped by a
    // branch), vectors laid out as load_pat's.
    template <int PAT>
    __device__ __forceinline__ static void load_guard(const Operand<T> &op, int o0, int k0, int K,
                                                      Vec (&st)[NV])
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int v = t + r * 256;
            const int o = PAT == PAT_OUTER ? (v % (R / VEC)) * VEC : v / (BK / VEC);
            const int kk = PAT == PAT_OUTER ? v / (R / VEC) : (v % (BK / VEC)) * VEC;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const long oe = o0 + o + (PAT == PAT_OUTER ? e : 0);
                const long ke = k0 + kk + (PAT == PAT_OUTER ? 0 : e);
                const bool in = oe < op.olim && ke < K;
                const long off = PAT == PAT_OUTER ? oe + ke * op.ld : ke + oe * op.ld;
                const T x = op.p[in ? off : 0];
                st[r][e] = in ? x : T(0);
            }
        }
    }

    template <int PAT, int LDS_LD>
    __device__ __forceinline__ static void store_pat(T (*s)[LDS_LD], const Vec (&st)[NV])
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int v = t + r * 256;
            if (PAT == PAT_KCONT) {
                const int kk = (v % (BK / VEC)) * VEC, o = v / (BK / VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) s[kk + e][o ^ lds_swz<T, R>(kk + e)] = st[r][e];
            } else {
                const int o = (v % (R / VEC)) * VEC, kk = v / (R / VEC);
                *(Vec *)&s[kk][o ^ lds_swz<T, R>(kk)] = st[r];
            }
        }
    }

    template <int LDS_LD>
    __device__ __forceinline__ static void store(T (*s)[LDS_LD], int pat, const Vec (&st)[NV])
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
            const int v = t + r * 256;
            if (pat == PAT_KCONT) {
                const int kk = (v % (BK / VEC)) * VEC, o = v / (BK / VEC);
#pragma unroll
                for (int e = 0; e < VEC; ++e) s[kk + e][o ^ lds_swz<T, R>(kk + e)] = st[r][e];
            } else {
                const int o = (v % (R / VEC)) * VEC, kk = v / (R / VEC);
                *(Vec *)&s[kk][o ^ lds_swz<T, R>(kk)] = st[r];
            }
        }
    }
};

template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef v4d Acc;
    __device__ __forceinline__ static Acc mma(double x, double y, Acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0);
    }
    // accumulator element r of lane l holds D[row][col] with
    // row = (l/16) + 4r, col = l%16 (D = C^T tile)
    __device__ __forceinline__ static int drow(int l, int r) { return (l >> 4) + 4 * r; }
};
template <> struct Mfma<float> {
    typedef v4f Acc;
    __device__ __forceinline__ static Acc mma(float x, float y, Acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
    }
    __device__ __forceinline__ static int drow(int l, int r) { return 4 * (l >> 4) + r; }
};

__device__ __forceinline__ void tri_decode(int b, int &hi, int &lo)
{
    // b-th pair (hi, lo) with hi >= lo in row-major order of a lower triangle
    int h = (int)((sqrt(8.0 * (double)b + 1.0) - 1.0) * 0.5);
    while (h * (h + 1) / 2 > b) --h;
    while ((h + 1) * (h + 2) / 2 <= b) ++h;
    hi = h;
    lo = b - h * (h + 1) / 2;
}

// C tile (tm, tn) of g: C = alpha*op(A)*op(B) + beta*C restricted to the
// tile (and to the triangle g.tri).  As / Bs: LDS staging of the caller.
// Ends with all waves past their last LDS read, so the caller may start
// another tile at once.
template <typename T, int BM, int BN, int BK>
__device__ __forceinline__ void gemm_tile(const GemmArgs<T> &g, int tm, int tn,
                                          T (*As)[BK][BM + 128 / sizeof(T)],
                                          T (*Bs)[BK][BN + 128 / sizeof(T)])
{
    constexpr int PAD = 128 / (int)sizeof(T);
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    typedef TileLoader<T, BM, BK> LA;
    typedef TileLoader<T, BN, BK> LB;
    typedef typename Mfma<T>::Acc Acc;

    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave & 1, wn = wave >> 1;

    Acc acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = Acc{};

    typename LA::Vec sa[LA::NV];
    typename LB::Vec sb[LB::NV];
    const int K = g.k;
    const int ktiles = (K + BK - 1) / BK;

    int pa = tile_pattern<T, BM, BK>(g.a, m0, 0, K);
    int pb = tile_pattern<T, BN, BK>(g.b, n0, 0, K);
    LA::load(g.a, m0, 0, K, pa, sa);
    LB::load(g.b, n0, 0, K, pb, sb);
    LA::template store<BM + PAD>(As[0], pa, sa);
    LB::template store<BN + PAD>(Bs[0], pb, sb);
    __syncthreads();

    for (int kt = 0; kt < ktiles; ++kt) {
        const int cur = kt & 1;
        const bool more = kt + 1 < ktiles;
        if (more) {
            const int k1 = (kt + 1) * BK;
            pa = tile_pattern<T, BM, BK>(g.a, m0, k1, K);
            pb = tile_pattern<T, BN, BK>(g.b, n0, k1, K);
            LA::load(g.a, m0, k1, K, pa, sa);
            LB::load(g.b, n0, k1, K, pb, sb);
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            T fa[FM], fb[FN];
            const int kr = kk + (lane >> 4);
            // (c0 + l) ^ swz = (c0 ^ shi) + (l ^ slo) for c0 a multiple of 16 and
            // l < 16: the high part of the swizzle depends on kk alone (a
            // constant of the unrolled loop), so the fragment offsets stay
            // immediate; the low part is one lane-dependent term per step
            static_assert(BM == BN, "one swizzle for both operands");
            const int shi = lds_swz<T, BM>(kk) & ~15;
            const int lo = (lane & 15) ^ (lds_swz<T, BM>(kr) & 15);
#pragma unroll
            for (int i = 0; i < FM; ++i)
                fa[i] = As[cur][kr][((wm * WM + i * 16) ^ shi) + lo];
#pragma unroll
            for (int j = 0; j < FN; ++j)
                fb[j] = Bs[cur][kr][((wn * WN + j * 16) ^ shi) + lo];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<T>::mma(fb[j], fa[i], acc[i][j]);
        }
        if (more) {
            LA::template store<BM + PAD>(As[cur ^ 1], pa, sa);
            LB::template store<BN + PAD>(Bs[cur ^ 1], pb, sb);
        }
        __syncthreads();
    }

    // Epilogue: accumulator (i, j) element r of this lane is C[row][col] with
    // row = m0 + wm*WM + i*16 + lane%16, col = n0 + wn*WN + j*16 + drow(lane, r).
    const T alpha = g.alpha, beta = g.beta;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const long gi = m0 + wm * WM + i * 16 + (lane & 15);
        if (gi >= g.m) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const long gj = n0 + wn * WN + j * 16 + Mfma<T>::drow(lane, r);
                if (gj >= g.n) continue;
                if (g.tri == SYM_LOWER && gi < gj) continue;
                if (g.tri == SYM_UPPER && gi > gj) continue;
                T *c = g.C + gi + gj * g.ldc;
                T v = alpha * acc[i][j][r];
                if (beta != T(0)) v += beta * *c;
                *c = v;
            }
        }
    }
}

// Fragments of one k step of 4 from a staged k-tile, and the products of one
// step: lane l of a wave holds row l%16 (of each 16-row block) at k = kk + l/16.
template <typename T, int BM, int BN, int BK>
struct TileMath {
    static constexpr int PAD = 128 / (int)sizeof(T);
    static constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    typedef typename Mfma<T>::Acc Acc;

    __device__ __forceinline__ static void fetch(const T (*A)[BM + PAD], const T (*B)[BN + PAD],
                                                 int kk, T (&fa)[FM], T (&fb)[FN])
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int wm = wave & 1, wn = wave >> 1, kr = kk + (lane >> 4);
        // (c0 + l) ^ swz = (c0 ^ high) + (l ^ low) for c0 a multiple of 16 and
        // l < 16: the high part of the swizzle depends on kk alone (a
        // constant of the unrolled loop), so the fragment offsets stay
        // immediate; the low part is one lane-dependent term per step
        const int ha = lds_swz<T, BM>(kk) & ~15, hb = lds_swz<T, BN>(kk) & ~15;
        const int la = (lane & 15) ^ (lds_swz<T, BM>(kr) & 15);
        const int lb = (lane & 15) ^ (lds_swz<T, BN>(kr) & 15);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = A[kr][((wm * WM + i * 16) ^ ha) + la];
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j] = B[kr][((wn * WN + j * 16) ^ hb) + lb];
    }
    __device__ __forceinline__ static void multiply(const T (&fa)[FM], const T (&fb)[FN],
                                                    Acc (&acc)[FM][FN])
    {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = Mfma<T>::mma(fb[j], fa[i], acc[i][j]);
    }
    // Accumulator (i, j) element r of this lane is C[row][col] with row = m0 +
    // wm*WM + i*16 + lane%16, col = n0 + wn*WN + j*16 + drow(lane, r); written
    // where row >= rlo, col >= clo, inside g and inside the triangle.  The 16
    // columns of a row block are read together before any of them is written
    // (one memory round trip per row block where beta is not 0); elements that
    // are not written read the tile's first one instead, so no load is skipped
    // by a branch.
    template <int TRI, bool BOUND>
    __device__ __forceinline__ static void finish(const GemmArgs<T> &g, int m0, int n0, int rlo,
                                                  int clo, const Acc (&acc)[FM][FN])
    {
        const bool inner = !BOUND && m0 == rlo && n0 == clo &&
                           (TRI == SYM_NONE || (TRI == SYM_LOWER ? m0 >= n0 + BN : n0 >= m0 + BM));
        if (inner) finish_part<TRI, BOUND, true>(g, m0, n0, rlo, clo, acc);
        else finish_part<TRI, BOUND, false>(g, m0, n0, rlo, clo, acc);
    }
    template <int TRI, bool BOUND, bool INNER>
    __device__ __forceinline__ static void finish_part(const GemmArgs<T> &g, int m0, int n0, int rlo,
                                                       int clo, const Acc (&acc)[FM][FN])
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int gi0 = m0 + (wave & 1) * WM + (lane & 15);
        const int gj0 = n0 + (wave >> 1) * WN + Mfma<T>::drow(lane, 0);
        constexpr int DR = sizeof(T) == 8 ? 4 : 1;  // columns from element r to r + 1
        const T alpha = g.alpha, beta = g.beta;
        T *const c0 = g.C + gi0 + (long)gj0 * g.ldc;
        const T *const any = g.C + rlo + (long)clo * g.ldc;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int gi = gi0 + i * 16;
            auto in = [&](int j, int r) {
                const int gj = gj0 + j * 16 + r * DR;
                return INNER || (gi >= rlo && gj >= clo && (!BOUND || (gi < g.m && gj < g.n)) &&
                                 (TRI == SYM_NONE || (TRI == SYM_LOWER ? gi >= gj : gi <= gj)));
            };
            T v[FN][4];
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] = alpha * acc[i][j][r];
            if (beta != T(0)) {
                T old[FN][4];
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        old[j][r] = *(in(j, r) ? c0 + i * 16 + (long)(j * 16 + r * DR) * g.ldc : any);
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[j][r] += beta * old[j][r];
            }
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (in(j, r)) c0[i * 16 + (long)(j * 16 + r * DR) * g.ldc] = v[j][r];
        }
    }
};

// Leading dimensions that the fast tile's 32-bit lane offsets reach: a lane is at
// most 31 (FP32: 63) columns and 32 elements from its tile's scalar address, 63 * 4 *
// 2^24 + 128 < 2^32.  Longer ones take 64-bit offsets.
constexpr long FAST_LD_MAX = 1l << 24;

// The fast tile's shapes.  NST: k-tiles of one operand on their way in registers.
// A 32 x 32 FP32 tile takes 32 of k at a time, one 16-byte load per thread.
template <typename T, int S> struct FastShape {
    static constexpr int BM = S, BN = S == 128 && sizeof(T) == 8 ? 64 : S;
    static constexpr int BK = S == 32 && sizeof(T) == 4 ? 32 : 16;
    static constexpr int NST = (S == 128 && sizeof(T) == 8) || BK == 32 ? 2 : 4;
    static constexpr int LDA = BM + 128 / (int)sizeof(T), LDB = BN + 128 / (int)sizeof(T);
};

// C tile (tm, tn) of g with access patterns PA / PB fixed at compile time, for
// m >= BM and n >= BN.  The last tile of a ragged dimension is moved back to
// end at the matrix's edge: it recomputes a few rows (columns) of its
// neighbour and does not store them, so every load is a full, unguarded
// vector load of any alignment.  Same k order and epilogue as gemm_tile, hence
// the same bits.
//
// Pipeline (bound: the matrix cores; LDS and memory have to stay out of their
// way): k-tiles t+2 ... t+1+NST travel from memory to registers while t is
// multiplied, t+1 is stored to the other LDS buffer during the first k step of t,
// and the fragments of a k step are read during the step before it -- across the
// one barrier of a k-tile too, which therefore sits in front of a step's products
// and not in front of its reads.  The barrier waits for LDS traffic alone.
// Measured, from reads in front of each step and guarded edge tiles over NST = 1 to
// the NST of FastShape: FP64 8192^3 NT 65.3, 68.0, 69.1 TFLOP/s; 2047 x 1531 x 1789
// TN on odd leading dimensions 44.4, 58.7, 65.6; FP32 4096^3 NN 121, 130, 137.
// NST is even: with an odd one the LDS buffer is no constant of the unrolled code
// (NST 3 was slower than 2).  128 x 128 FP64 tiles have no registers for a second
// stage; more than 256 registers a lane make the compiler move the accumulators to
// and from the accumulation registers in every k-tile (48 TFLOP/s).
template <typename T, int BM, int BN, int BK, int NST, int PA, int PB, int TRI, typename Off = unsigned>
__device__ __forceinline__ void gemm_fast_tile(const GemmArgs<T> &g, int tm, int tn,
                                               T (*As)[BK][BM + 128 / sizeof(T)],
                                               T (*Bs)[BK][BN + 128 / sizeof(T)])
{
    typedef TileMath<T, BM, BN, BK> M;
    typedef TileLoader<T, BM, BK> LA;
    typedef TileLoader<T, BN, BK> LB;
    constexpr int STEPS = BK / 4;
    static_assert(STEPS % 2 == 0, "the fragment buffers alternate over a k-tile");

    const int m0 = min(tm * BM, g.m - BM), n0 = min(tn * BN, g.n - BN);
    const int K = g.k, kfull = K / BK, ktiles = (K + BK - 1) / BK;
    const long lda = g.a.ld, ldb = g.b.ld;
    const T *pa = g.a.p + (PA == PAT_OUTER ? (long)m0 : (long)m0 * lda);
    const T *pb = g.b.p + (PB == PAT_OUTER ? (long)n0 : (long)n0 * ldb);
    const long stepa = PA == PAT_OUTER ? BK * lda : BK, stepb = PB == PAT_OUTER ? BK * ldb : BK;
    const Off va = LA::template voff<PA, Off>(lda), vb = LB::template voff<PB, Off>(ldb);

    typename M::Acc acc[M::FM][M::FN];
#pragma unroll
    for (int i = 0; i < M::FM; ++i)
#pragma unroll
        for (int j = 0; j < M::FN; ++j) acc[i][j] = typename M::Acc{};

    // k-tile t passes through register stage t % NST; pa / pb are uniform and
    // move on with the loads
    typename LA::Vec sa[NST][LA::NV];
    typename LB::Vec sb[NST][LB::NV];
    auto load_full = [&](int r) {
        LA::template load_pat<PA>(pa, lda, va, sa[r]);
        LB::template load_pat<PB>(pb, ldb, vb, sb[r]);
        pa += stepa;
        pb += stepb;
    };
    auto load_any = [&](int t, int r) {
        if (t < kfull) {
            load_full(r);
        } else if (t < ktiles) {
            LA::template load_ktail<PA, Off>(pa, lda, K - t * BK, sa[r]);
            LB::template load_ktail<PB, Off>(pb, ldb, K - t * BK, sb[r]);
        }
    };
    auto store = [&](int buf, int r) {
        LA::template store_pat<PA, BM + M::PAD>(As[buf], sa[r]);
        LB::template store_pat<PB, BN + M::PAD>(Bs[buf], sb[r]);
    };
    T fa[2][M::FM], fb[2][M::FN];

#pragma unroll
    for (int t = 0; t < NST; ++t) load_any(t, t);
    store(0, 0);
    load_any(NST, 0);
    lds_barrier();
    M::fetch(As[0], Bs[0], 0, fa[0], fb[0]);
    // k-tile kt out of buffer cur; kt + 1 leaves stage r for the other buffer
    int kt = 0;
    auto tile = [&](int cur, int r, bool steady) {
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            if (st + 1 < STEPS) {
                M::fetch(As[cur], Bs[cur], (st + 1) * 4, fa[(st + 1) & 1], fb[(st + 1) & 1]);
            } else {
                lds_barrier();
                M::fetch(As[cur ^ 1], Bs[cur ^ 1], 0, fa[0], fb[0]);
            }
            if (st == 0) {
                if (steady) {
                    store(cur ^ 1, r);
                    load_full(r);
                } else if (kt + 1 < ktiles) {
                    store(cur ^ 1, r);
                    load_any(kt + 1 + NST, r);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            M::multiply(fa[st & 1], fb[st & 1], acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        ++kt;
    };
    // U k-tiles per pass: buffer and stage are constants of the unrolled code
    constexpr int U = NST < 2 ? 2 : NST;
    static_assert(U % 2 == 0 && U % NST == 0, "a pass starts at buffer 0 and stage 1");
    while (kt + U + NST < kfull) {
#pragma unroll
        for (int q = 0; q < U; ++q) tile(q & 1, (q + 1) % NST, true);
    }
    while (kt < ktiles) {  // what is left: the ragged k-tile or nothing to load
#pragma unroll
        for (int q = 0; q < U; ++q)
            if (kt < ktiles) tile(q & 1, (q + 1) % NST, false);
    }
    M::template finish<TRI, false>(g, m0, n0, tm * BM, tn * BN, acc);
}

// The same tile where a dimension of C is smaller than the tile: every load
// guarded (load_guard) and the epilogue bounded; elements past an operand's
// end read as zero, as in gemm_tile, so the bits are still the same.
template <typename T, int BM, int BN, int BK, int PA, int PB>
__device__ __forceinline__ void gemm_edge_tile(const GemmArgs<T> &g, int tm, int tn,
                                               T (*As)[BK][BM + 128 / sizeof(T)],
                                               T (*Bs)[BK][BN + 128 / sizeof(T)])
{
    typedef TileMath<T, BM, BN, BK> M;
    typedef TileLoader<T, BM, BK> LA;
    typedef TileLoader<T, BN, BK> LB;
    const int m0 = tm * BM, n0 = tn * BN, K = g.k, ktiles = (K + BK - 1) / BK;
    typename M::Acc acc[M::FM][M::FN];
#pragma unroll
    for (int i = 0; i < M::FM; ++i)
#pragma unroll
        for (int j = 0; j < M::FN; ++j) acc[i][j] = typename M::Acc{};
    typename LA::Vec sa[LA::NV];
    typename LB::Vec sb[LB::NV];
    auto load = [&](int k0) {
        LA::template load_guard<PA>(g.a, m0, k0, K, sa);
        LB::template load_guard<PB>(g.b, n0, k0, K, sb);
    };
    auto store = [&](int buf) {
        LA::template store_pat<PA, BM + M::PAD>(As[buf], sa);
        LB::template store_pat<PB, BN + M::PAD>(Bs[buf], sb);
    };
    load(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < ktiles; ++kt) {
        const int cur = kt & 1;
        const bool more = kt + 1 < ktiles;
        if (more) load((kt + 1) * BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            T fa[M::FM], fb[M::FN];
            M::fetch(As[cur], Bs[cur], kk, fa, fb);
            M::multiply(fa, fb, acc);
        }
        if (more) store(cur ^ 1);
        __syncthreads();
    }
    M::template finish<SYM_NONE, true>(g, m0, n0, m0, n0, acc);
}

inline bool is_n(char c) { return c == 'N' || c == 'n'; }
inline bool is_l(char c) { return c == 'L' || c == 'l'; }
inline bool is_u(char c) { return c == 'U' || c == 'u'; }

template <typename T>
Operand<T> make_op(const T *p, long ld, int olim, int form, int sym)
{
    Operand<T> o;
    o.p = p;
    o.ld = ld;
    o.olim = olim;
    o.form = form;
    o.sym = sym;
    const int vec = 16 / (int)sizeof(T);
    o.vec_ok = (((uintptr_t)p & 15) == 0) && (ld % vec == 0);
    return o;
}

}  // namespace
