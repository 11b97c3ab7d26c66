// trsm_panel.hpp -- triangular solve of one panel of 16 right-hand sides on
// the FP64 matrix cores, shared by the per-call solves (trsm.hip) and the
// grouped ones of the serving loop (group.hip).
//
// One 512-thread workgroup solves op(T) X = alpha B for an order of at most
// 128 * SB, in blocks of 16 rows.  The four lower / upper, plain / transposed
// forms are one: the rows are numbered in the order in which they are solved,
// and op(T)(i, k) = A[i * si + k * sk], B(i, c) = B[i * ss + c * rs] with
// strides of either sign reach them.  FP32 operands are solved in FP64 and
// rounded once.
//
//  * Prologue: the 16 x 16 diagonal blocks are inverted in LDS, four per wave,
//    one lane per column, while the panel's loads are still in flight.  A block
//    whose inverse would cost accuracy (kInverseGrowth) stays as it is.
//  * Wave w keeps the sums of T[J, I] X_I over the solved blocks I for its blocks
//    J = w, w + 8, ... in MFMA accumulators.  When X of block st is published,
//    every wave adds T[J, st] X_st for its later blocks, the owner of block st + 1
//    that one first: it then forms X = inv(T_JJ) (B_J - sum) (the accumulator
//    layout is the operand layout), or substitutes where the block was left, and
//    publishes it.
//  * No barrier between steps: X_st is followed by a flag word in LDS, and a
//    wave waits for that word alone, so the chain of solves never waits for
//    the other blocks' updates.  The next owner reads word and X together (LDS
//    serves one wave's requests in order, so X is valid if the word was set).
//    All eight waves are resident and each publishes its blocks in increasing
//    order from words of lower blocks, so every wait ends.
//  * op(T) fragments are fetched DIST = 2 steps ahead (3 measured the same).
//
// Bound: per step the chain of 4 + 4 dependent v_mfma_f64_16x16x4 (64 cycles
// each) and two LDS trips: 0.7 us a block where barriers between the steps and
// substitution or an LDS wait before each read took 1.0 to 1.4.  Order 256, 4096
// right-hand sides: 14.5 us, 4 of them the loads and the inversion.
// Error of FP64 solves against 80-bit arithmetic, orders 64..2000, triangles whose
// diagonal outweighs their other entries: 1.0 to 2.7e-16 (substitution and
// recursion with products: 1.9 to 4.8e-16); FP32: 2.5e-8 up to order 512, 1.4e-7 at
// 2000 (1.4 to 3.2e-7).
#pragma once
#include "devcommon.hpp"
#include <type_traits>

namespace {

constexpr int TP_WAVES = 8, TP_THREADS = 64 * TP_WAVES;

// A product with the inverse Y of a block T can leave a residual far above that of
// a substitution.  How far shows in the inverse of the block scaled to a unit
// diagonal, Y_ij T_jj: a block with an entry beyond this limit is substituted.
// Residuals over random blocks, in units of u |T| |X| (substitution: up to 3):
// factors with a dominant diagonal, Cholesky factors and the L of a pivoted LU have
// entries up to 3 and leave 2 to 5; blocks within the limit 25 at most but for a few
// near bidiagonal ones (80); past it, off-diagonal entries to 2 beside a unit
// diagonal 600, entries to 4 1e5, the R of a 16-term monomial fit 2300.  FP32
// operands are solved in FP64: 2^20 times the limit is still far below their u.
template <typename IO> constexpr double kInverseGrowth = sizeof(IO) == 8 ? 4.0 : 4194304.0;

// LDS of one panel of order up to 128 * SB.
template <int SB>
struct PanelLds {
    // the solved rows; four rows are 32 banks apart modulo the 64, so a fragment
    // read (rows r, r + 4, ...) is free of conflicts
    double X[128 * SB][20];
    double L[8 * SB][16][17];  // diagonal blocks, then their inverses
    double R[8 * SB][16];      // reciprocals of the diagonal
    int kept[8 * SB];          // the block was not inverted: it is substituted
    int ready[8 * SB];         // X of the block is in place
    int odd;                   // a result that is not finite
};

struct PanelArgs {
    const void *A;    // op(T)(0, 0) in solve order
    void *B;          // row 0 of the panel's first right-hand side
    long si, sk;      // op(T)(i, k) = A[i * si + k * sk]
    long ss, rs;      // B(i, c) = B[i * ss + c * rs]
    int order, cols;  // cols <= 16 right-hand sides
    int unit;
    double alpha;
};

__device__ __forceinline__ void lds_order()
{
    __builtin_amdgcn_s_waitcnt(vm_wait(63) & ~(15 << 8));
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_wave_barrier();
}

// An LDS read that stays in program order with the other ones of its wave
// (a volatile one would also wait for its result before the next is issued).
__device__ __forceinline__ double lds_value(const double *p)
{
    return __builtin_bit_cast(double, __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP));
}

// |v| as an integer to compare (20 bits of the mantissa; a NaN is above all).
__device__ __forceinline__ unsigned magnitude(double v)
{
    return (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32) & 0x7fffffffu;
}

// f(0), f(1), ... f(N - 1) with compile-time arguments until one returns false
template <int S, int N, typename F> __device__ __forceinline__ void panel_steps(F &f)
{
    if constexpr (S < N) {
        if (f(std::integral_constant<int, S>{})) panel_steps<S + 1, N>(f);
    }
}

// One pass over the panel; the result is stored, and true returned, if it is finite
// or ALL.  KC: op(T)(i, k) is contiguous along k (|sk| = 1).  ALL: every diagonal
// block is substituted, with divisions, rows before a row left alone: for panels
// whose result is not finite, where a product with an inverse's zeros carries an
// infinity or a NaN of one row to the rows above it in the block, and a reciprocal
// may be infinite where the quotient is not.
template <typename IO, int SB, bool KC, bool ALL>
__device__ __forceinline__ bool panel_pass(const PanelArgs &p, PanelLds<SB> &s)
{
    constexpr int NBMAX = 8 * SB;               // blocks
    constexpr int PER = NBMAX * 256 / TP_THREADS;  // elements per thread: diagonal blocks, panel
    constexpr int DIST = 2;
    const IO *__restrict__ A = (const IO *)p.A;
    IO *B = (IO *)p.B;
    // (opaque, so that a caller's loop over panels keeps no address of this code
    // in registers across it: it spilled 240 of them)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    // (the wave number as a scalar: the branches on it are scalar branches, which
    // MFMA, blind to the lane mask, needs)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q0 = lane >> 4, cl = lane & 15;
    const int order = p.order, nb = (order + 15) / 16;
    const bool runs = p.ss == 1 || p.ss == -1;  // a right-hand side is contiguous

    if (tid < NBMAX) s.ready[tid] = 0;
    if (!ALL && tid == NBMAX) s.odd = 0;
    // Diagonal blocks first, the panel after them: loads complete in order, so
    // the inversion waits for the former alone.  A thread's elements are a fixed
    // step apart (every second block; 32 rows), so each kind takes one address
    // (order 512: 36.5 -> 35.4 us against an address per element).
    IO d[PER], v[PER];
    const int bk0 = tid >> 8, di = (tid >> 4) & 15, dk = tid & 15;
    const bool below = p.unit ? dk < di : dk <= di;
    auto in_diag = [&](int e) { return below && 16 * (bk0 + 2 * e) + di < order; };
    const long dstep = 32 * (p.si + p.sk);
    const IO *const dp = A + (16 * bk0 + di) * p.si + (16 * bk0 + dk) * p.sk;
#pragma unroll
    for (int e = 0; e < PER; ++e) d[e] = *(in_diag(e) ? dp + e * dstep : A);
    // contiguous along a right-hand side: 32 of its rows per pass; else 16 of a row
    const int pr = runs ? tid & 31 : tid >> 4, pc = runs ? tid >> 5 : tid & 15;
    auto in_panel = [&](int e) { return pr + 32 * e < order && pc < p.cols; };
    const long pstep = 32 * p.ss;
    const IO *const bp = B + pr * p.ss + pc * p.rs;
#pragma unroll
    for (int e = 0; e < PER; ++e) v[e] = *(in_panel(e) ? bp + e * pstep : B);
#pragma unroll
    for (int e = 0; e < PER; ++e)  // identity past the order
        s.L[bk0 + 2 * e][di][dk] = in_diag(e) ? (double)d[e] : di == dk ? 1.0 : 0.0;
    lds_barrier();
    if constexpr (!ALL) {
        // column cl of the inverse of block 4 * wave + q0; one division per lane
        // (16 of them in every lane took 1.5 us)
        const int bk = 4 * wave + q0;
        if (bk < nb && bk < NBMAX) {
            double y[16];
            const double own = 1.0 / s.L[bk][cl][cl];
            s.R[bk][cl] = own;
            const unsigned limit = magnitude(kInverseGrowth<IO> * own);
            lds_order();
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const double rc = s.R[bk][i];
                double t = i == cl ? 1.0 : 0.0;
#pragma unroll
                for (int k = 0; k < i; ++k) t = fma(-s.L[bk][i][k], y[k], t);
                y[i] = t * rc;
            }
            lds_order();  // every lane's reads of the block are done
            unsigned top = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) top = max(top, magnitude(y[i]));
            const bool kept = (__ballot(top > limit) >> (16 * q0) & 0xffff) != 0;
            if (cl == 0) s.kept[bk] = kept;
            if (__builtin_expect(!kept, 1))
#pragma unroll
                for (int i = 0; i < 16; ++i) s.L[bk][i][cl] = y[i];
        }
    }
#pragma unroll
    for (int e = 0; e < PER; ++e)
        s.X[pr + 32 * e][pc] = in_panel(e) ? p.alpha * (double)v[e] : 0.0;
    // op(T)[J, st] in MFMA A-operand layout for the wave's blocks J = wave + 8 q:
    // element u of a lane is op(T)(16 J + cl, 16 st + 4 q0 + u) -- the k order
    // that lets a lane read its four elements as one run where k is contiguous
    // (KC).  Rows past the order read the last one: they are finite where it is,
    // and reach nothing but the panel's rows past the order.
    const IO *row[SB];
#pragma unroll
    for (int q = 0; q < SB; ++q)
        row[q] = A + min(16 * (wave + TP_WAVES * q) + cl, order - 1) * p.si +
                 (KC && p.sk < 0 ? -(4 * q0 + 3) : 4 * q0 * p.sk);
    IO ring[DIST + 1][SB][4];
    auto fetch = [&](int st, IO (&f)[SB][4]) {
        const long k = 16l * min(st, nb - 2) * p.sk;
#pragma unroll
        for (int q = 0; q < SB; ++q)
            if (TP_WAVES * q + TP_WAVES - 1 > st) {
                if constexpr (KC) {
                    typedef IO Run __attribute__((ext_vector_type(4), aligned(sizeof(IO))));
                    const Run r = *(const Run *)(row[q] + k);
#pragma unroll
                    for (int u = 0; u < 4; ++u) f[q][u] = r[u];
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u) f[q][u] = row[q][k + u * p.sk];
                }
            }
    };
    // a run of stride -1 was read from its far end: element u is then k = 3 - u
    const int flip = KC && p.sk < 0 ? 3 : 0;
    if (nb > 1)
#pragma unroll
        for (int st = 0; st < DIST; ++st) fetch(st, ring[st]);
    lds_barrier();  // inverses and panel are in LDS (the fragments still on their way)

    // sums of op(T)[J, I] X_I, subtracted from B_J at the end: a running
    // difference would be rounded at B_J's size in every step.  (ALL: they start from
    // -B_J, as a sum may overflow where the difference does not.)
    v4d acc[SB];
#pragma unroll
    for (int q = 0; q < SB; ++q)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            acc[q][u] = ALL ? -s.X[16 * (wave + TP_WAVES * q) + q0 + 4 * u][cl] : 0.0;
    double inv[4], rhs[4];  // the inverse and B_J of the wave's next block to solve
    auto upcoming = [&](int q) {
        const int J = wave + TP_WAVES * q;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            inv[u] = ALL ? 0.0 : s.L[J][cl][4 * u + q0];
            rhs[u] = ALL ? 0.0 : s.X[16 * J + q0 + 4 * u][cl];
        }
    };
    upcoming(0);
    unsigned kept = ALL ? ~0u : 0u;  // bit q: the wave's block q is substituted
#pragma unroll
    for (int q = 0; q < SB; ++q) {
        const int J = wave + TP_WAVES * q;
        if (!ALL && J < nb) kept |= (unsigned)__builtin_amdgcn_readfirstlane(s.kept[J]) << q;
    }
    bool finite = true;
    // X_J = inv(T_JJ) B_J, published
    auto solve = [&](int q) {
        const int J = wave + TP_WAVES * q;
        v4d x = {0.0, 0.0, 0.0, 0.0};
        if (ALL || __builtin_expect(kept >> q & 1, 0)) {
            // substitution, row r in element r / 4 of the lanes with q0 = r % 4 (T is
            // zero above its diagonal)
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = rhs[u] - acc[q][u];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll 1
                for (int h = 0; h < 4; ++h) {
                    const int r = 4 * e + h;
                    const double b = __shfl(x[e], cl + 16 * h);
                    const double xr = ALL ? b / s.L[J][r][r] : b * s.R[J][r];
                    if (!ALL || q0 >= h)
                        x[e] = q0 == h ? xr : fma(-s.L[J][4 * e + q0][r], xr, x[e]);
#pragma unroll
                    for (int u = e + 1; u < 4; ++u) x[u] = fma(-s.L[J][4 * u + q0][r], xr, x[u]);
                }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                x = __builtin_amdgcn_mfma_f64_16x16x4f64(inv[u], rhs[u] - acc[q][u], x, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) s.X[16 * J + q0 + 4 * u][cl] = x[u];
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (lane == 0) __hip_atomic_store(&s.ready[J], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
        for (int u = 0; u < 4; ++u) finite = finite && __builtin_isfinite(x[u]);
        if (q + 1 < SB) upcoming(q + 1);
    };
    if (wave == 0) solve(0);
    const int last = min(nb, NBMAX) - 1;  // the wave's last block is at most this one
    const int mine = last - ((last - wave) & (TP_WAVES - 1));  // its last block (< 0: none)
    // one block's sum takes on op(T)[J, st] X_st
    auto update = [&](int q, const IO (&f)[4], const double (&x)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)f[u], x[u], acc[q], 0, 0, 0);
    };
    // step st, a compile-time constant: the fragment ring and the accumulators
    // stay in registers.  False once nothing of this wave waits for X_st.
    auto step = [&](auto stc) {
        constexpr int st = decltype(stc)::value, W = TP_WAVES;
        if (st >= mine) return false;
        if constexpr (st + DIST < NBMAX - 1) fetch(st + DIST, ring[(st + DIST) % (DIST + 1)]);
        IO(&f)[SB][4] = ring[st % (DIST + 1)];
        constexpr int qn = (st + 1) / W;  // block st + 1 at its owner
        double x[4];
        auto flag = [&] {
            return __builtin_amdgcn_readfirstlane(
                __hip_atomic_load(&s.ready[st], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        };
        auto read_x = [&] {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                x[u] = lds_value(&s.X[16 * st + 4 * q0 + (u ^ flip)][cl]);
        };
        if (wave == (st + 1) % W) {
            // ahead of the other wave of this SIMD until X is out: its trailing
            // updates would take every second slot of the matrix core
            __builtin_amdgcn_s_setprio(3);
            int ok;
            do {
                ok = __hip_atomic_load(&s.ready[st], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                read_x();
            } while (!__builtin_amdgcn_readfirstlane(ok));
            update(qn, f[qn], x);
            solve(qn);
            __builtin_amdgcn_s_setprio(0);
        } else {
            while (!flag()) __builtin_amdgcn_s_sleep(1);
            read_x();
            if (wave + W * qn > st + 1) update(qn, f[qn], x);
        }
#pragma unroll
        for (int q = qn + 1; q < SB; ++q) update(q, f[q], x);
        return true;
    };
    panel_steps<0, NBMAX - 1>(step);
    if (!ALL && __any(!finite) && lane == 0) s.odd = 1;
    __syncthreads();  // all of X, and whether it is finite
    if (!ALL && __builtin_amdgcn_readfirstlane(s.odd)) return false;
    // (the thread's place in the panel once more: kept over the steps it would cost
    // the registers of a third workgroup per CU where SB is 1)
    int out = threadIdx.x;
    asm volatile("" : "+v"(out));
    const int orow = runs ? out & 31 : out >> 4, ocol = runs ? out >> 5 : out & 15;
    IO *const op = B + orow * p.ss + ocol * p.rs;
#pragma unroll
    for (int e = 0; e < PER; ++e)
        if (orow + 32 * e < order && ocol < p.cols) op[e * pstep] = (IO)s.X[orow + 32 * e][ocol];
    return true;
}

// A panel whose result is not finite takes a second pass, from the right-hand sides
// that are still in memory.  Order 512, 4096 right-hand sides, finite 50.6 us; a zero
// pivot or NaNs 164 us (979 by plain substitution, row by row, from global memory).
template <typename IO, int SB, bool KC>
__device__ __forceinline__ void trsm_panel(const PanelArgs &p, PanelLds<SB> &s)
{
    if (__builtin_expect(!panel_pass<IO, SB, KC, false>(p, s), 0)) panel_pass<IO, SB, KC, true>(p, s);
}

// Panel arguments of op(T) X = alpha B: T lower (`lower`) in plain or transposed
// storage (transN: op(T)(i, k) = A[i + k * lda]), rows of B `ss` apart.
template <typename IO>
__device__ __forceinline__ PanelArgs panel_args(const IO *A, long lda, int transN, int lower,
                                                int unit, IO *B, long ss, long rs, int order,
                                                int cols, double alpha)
{
    PanelArgs p;
    p.si = transN ? 1 : lda;
    p.sk = transN ? lda : 1;
    p.ss = ss;
    p.rs = rs;
    p.A = A;
    p.B = B;
    if (!lower) {  // upper: solved from the last row up
        p.A = A + (long)(order - 1) * (1 + lda);
        p.B = B + (order - 1) * ss;
        p.si = -p.si;
        p.sk = -p.sk;
        p.ss = -ss;
    }
    p.order = order;
    p.cols = cols;
    p.unit = unit;
    p.alpha = alpha;
    return p;
}

}  // namespace
