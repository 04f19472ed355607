// qpc_solve.hip -- partitioned banded CN solves, their tables and the
// time-batched factorisation of the coupling sweeps (gfx950), built for band
// half-widths p = 7 and p = 8 (template parameter P).
#include "qpc_solve.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

namespace qpc {
namespace {

// a + t x with fused multiply-adds (4 for complex t, 2 for real t)
__device__ inline cplx tmac(cplx a, cplx t, cplx x) {
    return {fma(-t.im, x.im, fma(t.re, x.re, a.re)), fma(t.im, x.re, fma(t.re, x.im, a.im))};
}
__device__ inline cplx tmac(cplx a, double t, cplx x) { return {fma(t, x.re, a.re), fma(t, x.im, a.im)}; }
// a - t x with fused multiply-adds (4 for complex t, 2 for real t)
__device__ inline cplx tmsub(cplx a, cplx t, cplx x) {
    return {fma(t.im, x.im, fma(-t.re, x.re, a.re)), fma(-t.im, x.re, fma(-t.re, x.im, a.im))};
}
__device__ inline cplx tmsub(cplx a, double t, cplx x) { return {fma(-t, x.re, a.re), fma(-t, x.im, a.im)}; }
__device__ inline cplx tmulf(cplx a, cplx b) {
    return {fma(-a.im, b.im, a.re * b.re), fma(a.im, b.re, a.re * b.im)};
}
// a complex number in LDS: 16-byte aligned, so that it moves in one access
struct alignas(16) lcplx {
    double re, im;
    __device__ operator cplx() const { return {re, im}; }
};
__device__ inline lcplx lc(cplx a) { return {a.re, a.im}; }
__device__ inline double tzero(double) { return 0.0; }
__device__ inline cplx tzero(cplx) { return {0.0, 0.0}; }
__device__ inline double tone(double) { return 1.0; }
__device__ inline cplx tone(cplx) { return {1.0, 0.0}; }

// The two table formats (qpc_solve.h) in units of 16 bytes: UF units per row
// and direction, `row` units per row, the backward ones from unit boff on.
// coef(c, k): the coefficient k = 1..P of a row's units; diag: its diagonal.
template <class TF, int P>
struct TabFmt;
template <int P>
struct TabFmt<double, P> {
    static constexpr bool SYM = false;
    static constexpr int UF = real_units(P), row = 2 * UF, boff = UF;
    __host__ __device__ static int64_t units(const Geom& g) { return g.tab_elems / 2; }
    __host__ __device__ static int64_t trf_elems(const Geom& g) { return g.trf_elems; }
    __device__ static double coef(const cplx (&c)[UF], int k) { return k & 1 ? c[(k - 1) / 2].re : c[(k - 1) / 2].im; }
    __device__ static double diag(const cplx (&c)[UF]) { return P & 1 ? c[UF - 1].im : c[UF - 1].re; }
};
template <int P>
struct TabFmt<cplx, P> {
    static constexpr bool SYM = true;
    static constexpr int UF = P + 1, row = P + 1, boff = 0;
    __host__ __device__ static int64_t units(const Geom& g) { return g.ctab_elems; }
    __host__ __device__ static int64_t trf_elems(const Geom& g) { return g.ctrf_elems; }
    __device__ static cplx coef(const cplx (&c)[UF], int k) { return c[k - 1]; }
    __device__ static cplx diag(const cplx (&c)[UF]) { return c[P]; }
};
// first unit of partition g's column in a table
template <class TF, int P>
__device__ inline int64_t part_col(int g) {
    return (int64_t)(g >> 6) * kPM * TabFmt<TF, P>::row * kLane + (g & 63);
}
// its byte offset
template <class TF, int P>
__device__ inline unsigned part_off(int g) {
    return (unsigned)part_col<TF, P>(g) * 16u;
}
// the units of one direction of a real row from its coefficients 1..P and diagonal
template <int P>
__device__ inline void put_real(cplx* o, const double* f, double d) {
#pragma unroll
    for (int u = 0; u < P / 2; ++u) o[(int64_t)u * kLane] = cplx{f[2 * u], f[2 * u + 1]};
    o[(int64_t)(real_units(P) - 1) * kLane] = P & 1 ? cplx{f[P - 1], d} : cplx{d, 0.0};
}
// 16 bytes per lane from global memory straight into LDS (to + lane), and the
// wait for all of them
__device__ inline void lds_load16(const cplx* from, lcplx* to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                     (__attribute__((address_space(3))) void*)to, 16, 0, 0);
}
__device__ inline void lds_load_wait() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

__device__ inline int table_of(const TabMap& tm, int ch) {
    if (tm.mode == 4) return tm.map[ch] & kMapIdx;
    if (tm.mode == 1) return 0;
    if (tm.mode == 3) return ch % tm.L;
    if (tm.mode == 2) {
        const int im = ch / tm.L, il = ch % tm.L;
        const int m = im + tm.m0;
        return il + (m < 0 ? -m : m);
    }
    return ch;
}

// a channel whose operator is the complex conjugate of its table's (mode 4):
// it is solved as conj(A^-1 B conj(z)), the table's own arithmetic on the
// conjugated input with its scalar, then conjugated
__device__ inline bool conj_of(const TabMap& tm, int ch) { return tm.mode == 4 && (tm.map[ch] & kMapConj); }
__device__ inline cplx cj_if(bool c, cplx v) { return c ? cplx{v.re, -v.im} : v; }

// ---------------------------------------------------------------------------
// Right-hand sides.  Their loads are unconditional, from indices clamped
// into [0, N), and band entries outside the matrix are zero (stored zero, or
// zeroed after loading), so every load of a row is in flight at once: a load
// under a branch compiles to a load-and-wait pair.  The sums keep their
// order; the extra terms add exact zeros.

// entry i of diagonal j: a uniform address per diagonal and one offset
template <class T>
__device__ inline T diag_at(const T* D, int j, int N, int i) {
    return *(const T*)((const char*)(D + (int64_t)j * N) + (unsigned)i * (unsigned)sizeof(T));
}

// Row i < N of a per-table complex band (diagonal-major, B(i, i+k) =
// U[k*N + i], zero where i + k >= N): its entries, then (B z)_i from
// z(d) = z_{i+d}, |d| <= P
template <int P>
struct CBandRow {
    cplx ul[P], uu[P + 1];
    __device__ inline void load(const cplx* __restrict__ U, int i, int N) {
#pragma unroll
        for (int j = 1; j <= P; ++j) ul[j - 1] = diag_at(U, j, N, max(i - j, 0));
#pragma unroll
        for (int k = 0; k <= P; ++k) uu[k] = diag_at(U, k, N, i);
    }
    // explicit fused multiply-adds, so that every kernel forming the row
    // rounds it alike (a complex product leaves the contraction open)
    template <class Z>
    __device__ inline cplx apply(Z z, int i) const {
        cplx v = {0.0, 0.0};
#pragma unroll
        for (int j = 1; j <= P; ++j) {
            const cplx u = i - j >= 0 ? ul[j - 1] : cplx{0.0, 0.0};
            v = tmac(v, u, z(-j));
        }
#pragma unroll
        for (int k = 0; k <= P; ++k) v = tmac(v, uu[k], z(k));
        return v;
    }
};

// Row i < N of the bands shared by every channel: the mask, or for the
// RHS_SX_* kinds S and X, whose entries come in {S, X} pairs (one load for
// both).  Lower entries B(i, i-j) = D[j][i-j] (zero above the first row),
// upper B(i, i+k) = D[k][i] (stored zero where i + k >= N).
template <int RHS, int P>
struct SBandRow {
    static constexpr bool SX = RHS != RHS_RBAND;
    double sl[P], su[P + 1], xl[P], xu[P + 1];
    __device__ inline void load(const RhsArgs& ra, int i, int N) {
#pragma unroll
        for (int j = 1; j <= P; ++j) {
            if constexpr (SX) {
                const cplx q = diag_at(ra.sx, j, N, max(i - j, 0));
                sl[j - 1] = q.re;
                xl[j - 1] = q.im;
            } else {
                sl[j - 1] = diag_at(ra.rband, j, N, max(i - j, 0));
                xl[j - 1] = 0.0;
            }
        }
#pragma unroll
        for (int k = 0; k <= P; ++k) {
            if constexpr (SX) {
                const cplx q = diag_at(ra.sx, k, N, i);
                su[k] = q.re;
                xu[k] = q.im;
            } else {
                su[k] = diag_at(ra.rband, k, N, i);
                xu[k] = 0.0;
            }
        }
#pragma unroll
        for (int j = 1; j <= P; ++j)
            if (i - j < 0) sl[j - 1] = xl[j - 1] = 0.0;
    }
    // (B z)_i from z(d) = z_{i+d}, |d| <= P; e = eig * ifdt of the channel
    template <class Z>
    __device__ inline cplx apply(Z z, double e) const {
        cplx sz = {0.0, 0.0}, zl = {0.0, 0.0}, zu = {0.0, 0.0};
#pragma unroll
        for (int j = 1; j <= P; ++j) {
            const cplx v = z(-j);
            sz += sl[j - 1] * v;
            if (SX) zl += xl[j - 1] * v;
        }
#pragma unroll
        for (int k = 0; k <= P; ++k) {
            const cplx v = z(k);
            sz += su[k] * v;
            if (SX) zu += xu[k] * v;
        }
        if (RHS == RHS_SX_SYM) {
            // a = S - ifet X with ifet = i*e:  v = Sz - i e (Xz)
            const cplx xz = zl + zu;
            return {sz.re + e * xz.im, sz.im - e * xz.re};
        } else if (RHS == RHS_SX_ASY) {
            // a = S + e X (lower) and S - e X (upper), e real
            return {sz.re + e * (zl.re - zu.re), sz.im + e * (zl.im - zu.im)};
        }
        return sz;
    }
};

// ---------------------------------------------------------------------------
// One table row of one partition and direction in registers (UF units).
// Forward (acc[k]: what the rows above contribute to row s + k): the row's value
// is its right-hand side v with what it has gathered, its multiples go to the P
// rows below, and row s + P enters with nothing.  The state a partition hands on
// is what its rows contribute to the first P rows of the next.
//
// The right-hand side comes last for the sake of its rounding: the farthest
// rows' products are the first to be added, and a sum that began with v would
// round each of them at v's size.  Errors of a free / mask solve of N = 240 (p =
// 7) against 80-bit arithmetic: 1.24e-14 / 2.52e-14; with v first 1.42e-14 /
// 3.32e-14; with v first and the nearest row's product next 1.23e-14 / 2.49e-14,
// but then every product waits for the row above.  Launches take the same time
// to 0.5%.
template <class TF, int P>
__device__ inline cplx fwd_row(const cplx (&c)[TabFmt<TF, P>::UF], cplx v, cplx (&acc)[P]) {
    using F = TabFmt<TF, P>;
    const cplx z = {v.re + acc[0].re, v.im + acc[0].im};
    cplx y;  // what the lower rows' updates take, and the stored row
    if constexpr (F::SYM) y = z;
    else y = {F::diag(c) * z.re, F::diag(c) * z.im};
#pragma unroll
    for (int k = 1; k < P; ++k) acc[k - 1] = tmsub(acc[k], F::coef(c, k), y);
    acc[P - 1] = tmsub(cplx{0.0, 0.0}, F::coef(c, P), y);
    if constexpr (F::SYM) return tmulf(F::diag(c), z);
    else return y;
}
// Backward (state h[k] = x_{s+1+k}): x_s from the stored row, oldest term
// first, so that only the last product waits for x_{s+1}
template <class TF, int P>
__device__ inline cplx bwd_row(const cplx (&c)[TabFmt<TF, P>::UF], cplx y, cplx (&h)[P]) {
    using F = TabFmt<TF, P>;
    cplx x = y;
    if constexpr (!F::SYM) x = {F::diag(c) * y.re, F::diag(c) * y.im};
#pragma unroll
    for (int k = P; k >= 1; --k) x = tmsub(x, F::coef(c, k), h[k - 1]);
#pragma unroll
    for (int k = P - 1; k > 0; --k) h[k] = h[k - 1];
    h[0] = x;
    return x;
}

// ---------------------------------------------------------------------------
// Rows of a partition are taken in blocks of RB.  The units of the block in
// hand sit in registers; as soon as a row is done its registers are filled
// with the same row of the next block, so that a block's loads are in flight
// while the block before runs.  Blocks [LB0, LB1) of a staged work-group come
// from LDS, the others from the table.  The block loops stay rolled and there
// is no branch between rows: a branch costs a wave about as much as six FP64
// operations, and code that is not in the instruction cache costs twice its
// run time, so the solves of a step together must stay within it (64 KB).
template <class TF, int P>
struct Blocks {
    static constexpr int RB = 4, NB = kPM / RB;
    static constexpr int LB0 = 1, LB1 = P == 7 ? 4 : 3;  // what the LDS holds beside the rows and states
    static constexpr int LR = (LB1 - LB0) * RB;          // staged rows
    static constexpr int UF = TabFmt<TF, P>::UF, UT = TabFmt<TF, P>::row;
    static_assert(kPM % RB == 0, "a pass is a whole number of blocks");
};
template <class TF, int P>
using RowRegs = cplx[TabFmt<TF, P>::UF];
template <class TF, int P>
using BlockRegs = RowRegs<TF, P>[Blocks<TF, P>::RB];

// unit k of the run at base (uniform), this lane's byte offset off
__device__ inline cplx unit_at(const cplx* base, unsigned off, int k) {
    return *(const cplx*)((const char*)(base + (int64_t)k * kLane) + off);
}
// UN units of row r of the block at p
template <class TF, int P, int UN>
__device__ inline void row_g(RowRegs<TF, P>& c, const cplx* p, unsigned off, int r) {
#pragma unroll
    for (int u = 0; u < UN; ++u) c[u] = unit_at(p, off, r * TabFmt<TF, P>::row + u);
}
template <class TF, int P, int UN>
__device__ inline void block_g(BlockRegs<TF, P>& c, const cplx* p, unsigned off) {
#pragma unroll
    for (int r = 0; r < Blocks<TF, P>::RB; ++r) row_g<TF, P, UN>(c[r], p, off, r);
}

// The row buffer: kRowStride slots per partition (an odd count, so that lanes
// of consecutive partitions fall on different banks), row s of slot ln at
// ln * kRowStride + s; kRowPad slots on either side for the passes' read-ahead
constexpr int kRowStride = kPM + 1, kRowPad = 4;
constexpr int kRowSlots = kLane * kRowStride + 2 * kRowPad;
__device__ inline int row_slot(int s, int ln) { return kRowPad + ln * kRowStride + s; }

// the rows of one block, written to wb[r]; the block's registers are refilled
// from LDS (l: this lane's units) or the table (p), v[r] from the next block's
// rows at nv
template <class TF, int P, bool L>
__device__ inline void fwd_block(BlockRegs<TF, P>& c, cplx (&v)[Blocks<TF, P>::RB], const lcplx* nv, lcplx* wb,
                                 const lcplx* l, const cplx* p, unsigned off, cplx (&acc)[P]) {
    using B = Blocks<TF, P>;
#pragma unroll
    for (int r = 0; r < B::RB; ++r) {
        const cplx y = fwd_row<TF, P>(c[r], v[r], acc);
        v[r] = nv[r];
        wb[r] = lc(y);
#pragma unroll
        for (int u = 0; u < B::UF; ++u)
            c[r][u] = L ? (cplx)l[(r * B::UF + u) * kLane] : unit_at(p, off, r * B::UT + u);
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <class TF, int P, bool L>
__device__ inline void bwd_block(BlockRegs<TF, P>& c, cplx (&v)[Blocks<TF, P>::RB], const lcplx* rb, lcplx* wb,
                                 const lcplx* l, const cplx* p, unsigned off, cplx (&h)[P]) {
    using B = Blocks<TF, P>;
    constexpr int UB = TabFmt<TF, P>::SYM ? P : B::UF;  // a symmetric row's diagonal is not read
#pragma unroll
    for (int r = B::RB - 1; r >= 0; --r) {
        const cplx x = bwd_row<TF, P>(c[r], v[r], h);
        v[r] = rb[r - B::RB];
        wb[r] = lc(x);
#pragma unroll
        for (int u = 0; u < UB; ++u)
            c[r][u] = L ? (cplx)l[(r * B::UF + u) * kLane] : unit_at(p, off, r * B::UT + u);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One pass over the rows of slot ln (rows: its first row; T: the direction's
// units of the table, uniform).  c holds the first block at entry and the
// block at `after` at the end.  Rows are written to `out` (their own place, or
// a scrap block of RB rows when ostep is 0).
template <class TF, int P, bool STAGED>
__device__ inline void fwd_pass(BlockRegs<TF, P>& c, const cplx* T, unsigned off, const lcplx* sL,
                                const lcplx* rows, lcplx* out, int ostep, cplx (&acc)[P], const cplx* after) {
    using B = Blocks<TF, P>;
    cplx v[B::RB];
#pragma unroll
    for (int r = 0; r < B::RB; ++r) v[r] = rows[r];
    if constexpr (STAGED) {
#pragma unroll 1
        for (int i = 0; i < B::LB1 - B::LB0; ++i) {
            rows += B::RB;
            fwd_block<TF, P, true>(c, v, rows, out, sL, nullptr, 0, acc);
            out += ostep;
            sL += B::RB * B::UF * kLane;
        }
    }
    constexpr int G0 = STAGED ? B::LB1 : 1, GN = B::NB + 1 - G0;  // the blocks still to load: G0 .. NB-1, after
    T += (int64_t)G0 * B::RB * B::UT * kLane;
#pragma unroll 1
    for (int i = 0; i < GN; ++i) {
        rows += B::RB;
        fwd_block<TF, P, false>(c, v, rows, out, nullptr, i == GN - 1 ? after : T, off, acc);
        out += ostep;
        T += B::RB * B::UT * kLane;
    }
}
template <class TF, int P, bool STAGED>
__device__ inline void bwd_pass(BlockRegs<TF, P>& c, const cplx* T, unsigned off, const lcplx* sL,
                                const lcplx* rows, lcplx* out, int ostep, cplx (&h)[P], const cplx* after) {
    using B = Blocks<TF, P>;
    cplx v[B::RB];
    rows += (B::NB - 1) * B::RB;
    out += (ostep ? B::NB - 1 : 0) * B::RB;
#pragma unroll
    for (int r = 0; r < B::RB; ++r) v[r] = rows[r];
    sL += (B::LR - B::RB) * B::UF * kLane;
    int b = B::NB - 2;  // the block to load next
#pragma unroll 1
    for (int ph = 0; ph < 2; ++ph) {
        const int stop = STAGED && ph == 0 ? B::LB1 : -1;
#pragma unroll 1
        for (; b >= stop; --b) {
            bwd_block<TF, P, false>(c, v, rows, out, nullptr, b < 0 ? after : T + b * (B::RB * B::UT * kLane), off, h);
            rows -= B::RB;
            out -= ostep;
        }
        if constexpr (!STAGED) break;
        if (ph == 0) {
#pragma unroll 1
            for (; b >= B::LB0; --b) {
                bwd_block<TF, P, true>(c, v, rows, out, sL, nullptr, 0, h);
                rows -= B::RB;
                out -= ostep;
                sL -= B::RB * B::UF * kLane;
            }
        }
    }
}

// The incoming state of every partition from the pass-A end states E and the
// partitions' own transfer matrices: s_g <- E_g + T_g s_{g-1} (g+1 backward),
// PK - 1 times from s = E, so that s_{g-1} holds the PK partitions before g,
// the same sums as Horner's rule over them.  A matrix is read once and stays
// in registers; only states pass between lanes, through LDS: entry r of slot
// ln at r * kSt + ln, with a column of zeros after the slots for the neighbour
// that does not exist.
constexpr int kSt = kLane + 1;
constexpr int kWavesStaged = 8, kHelp = kWavesStaged - 1;

// entry (r, c) of the direction's matrix, T the table's set (uniform); a
// symmetric table's backward matrix is the transpose of its forward one
template <class TF, int P>
__device__ inline unsigned trf_off(int g) {
    return ((unsigned)(g >> 6) * (TabFmt<TF, P>::SYM ? 1 : 2) * P * P * kLane + (g & 63)) * (unsigned)sizeof(TF);
}
template <class TF, int P>
__device__ inline TF trf_at(const TF* T, unsigned off, int dir, int r, int c) {
    constexpr bool SYM = TabFmt<TF, P>::SYM;
    const int e = SYM ? (dir ? c * P + r : r * P + c) : dir * P * P + r * P + c;
    return *(const TF*)((const char*)(T + (int64_t)e * kLane) + off);
}
// the column of slot ln's neighbour
__device__ inline int neighbour(int ln, int n, int dir) {
    const int nb = dir == 0 ? ln - 1 : ln + 1;
    return nb >= 0 && nb < n ? nb : kLane;
}

// one wave: slot ln of n; e enters as the end states and leaves as the
// incoming state
template <class TF, int P>
__device__ inline void carry1(const TF (&t)[P][P], lcplx* sS, int ln, int n, int dir, int PK, cplx (&e)[P]) {
    const int q = neighbour(ln, n, dir);
#pragma unroll
    for (int r = 0; r < P; ++r) sS[r * kSt + ln] = lc(e[r]);
    __syncthreads();
#pragma unroll 1
    for (int k = 1; k < PK; ++k) {
        cplx in[P];
#pragma unroll
        for (int c = 0; c < P; ++c) in[c] = sS[c * kSt + q];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < P; ++r) {
            cplx a = e[r];
#pragma unroll
            for (int c = 0; c < P; ++c) a = tmac(a, t[r][c], in[c]);
            sS[r * kSt + ln] = lc(a);
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < P; ++r) e[r] = sS[r * kSt + q];
    __syncthreads();
}

// a staged work-group: the helper waves share the rows of the product (helper
// hw has row hw, and hw + 7 of eight), wave 0 waits.  One barrier per step.
constexpr int trf_rows(int P) { return (P + kHelp - 1) / kHelp; }
template <class TF, int P>
__device__ inline void carry_load(TF (&t)[trf_rows(P)][P], const TF* T, unsigned off, int dir, int hw) {
#pragma unroll
    for (int i = 0; i < trf_rows(P); ++i)
#pragma unroll
        for (int c = 0; c < P; ++c) t[i][c] = trf_at<TF, P>(T, off, dir, min(hw + kHelp * i, P - 1), c);
}
template <class TF, int P>
__device__ inline void carry8(const TF (&t)[trf_rows(P)][P], const lcplx* sE, lcplx* sS, int ln, int n, int dir, int PK,
                              int hw) {
    const int q = neighbour(ln, n, dir);
    cplx e[trf_rows(P)];
#pragma unroll
    for (int i = 0; i < trf_rows(P); ++i) e[i] = sE[min(hw + kHelp * i, P - 1) * kSt + ln];
    const lcplx* src = sE;
#pragma unroll 1
    for (int k = 1; k < PK; ++k) {
        lcplx* dst = sS + (k & 1) * P * kSt;
        cplx in[P];
#pragma unroll
        for (int c = 0; c < P; ++c) in[c] = src[c * kSt + q];
#pragma unroll
        for (int i = 0; i < trf_rows(P); ++i) {
            const int r = min(hw + kHelp * i, P - 1);  // (a row past the last repeats the last)
            cplx a = e[i];
#pragma unroll
            for (int c = 0; c < P; ++c) a = tmac(a, t[i][c], in[c]);
            dst[r * kSt + ln] = lc(a);
        }
        __syncthreads();
        src = dst;
    }
}
// the buffer that holds the result after PK - 1 steps
template <int P>
__device__ inline const lcplx* carried(const lcplx* sE, const lcplx* sS, int PK) {
    return PK > 1 ? sS + ((PK - 1) & 1) * P * kSt : sE;
}

template <int... I, class F>
__device__ inline void each(std::integer_sequence<int, I...>, F f) {
    (f(std::integral_constant<int, I>{}), ...);
}

// v = B z for per-table bands (RHS_CBAND), one lane per (row, channel)
template <int P>
__global__ __launch_bounds__(256) void k_rhs(RhsArgs ra, TabMap tm, const cplx* __restrict__ zin,
                                             cplx* __restrict__ vout, int N) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int ch = blockIdx.y;
    if (i >= N) return;
    CBandRow<P> b;
    b.load(ra.cband + (int64_t)table_of(tm, ch) * (P + 1) * N, i, N);
    const cplx* z = zin + (int64_t)ch * N;
    vout[(int64_t)ch * N + i] = b.apply([&](int d) { return z[min(max(i + d, 0), N - 1)]; }, i);
}

// v = B z for bands shared by every channel (RHS_RBAND, RHS_SX_*): a lane
// loads the band entries of its row once and applies them to kRhsCG channels
// (2 measured fastest: 4 keeps too many loads live, 1 repeats the band loads)
constexpr int kRhsCG = 2;
template <int RHS, int P>
__global__ __launch_bounds__(256) void k_rhs_shared(RhsArgs ra, const cplx* __restrict__ zin,
                                                    cplx* __restrict__ vout, int N, int nch) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    SBandRow<RHS, P> b;
    b.load(ra, i, N);
#pragma unroll
    for (int c = 0; c < kRhsCG; ++c) {
        const int ch = blockIdx.y * kRhsCG + c;
        if (ch < nch) {
            const cplx* z = zin + (int64_t)ch * N;
            const double e = SBandRow<RHS, P>::SX ? ra.eig[ch] * ra.ifdt : 0.0;
            vout[(int64_t)ch * N + i] = b.apply([&](int d) { return z[min(max(i + d, 0), N - 1)]; }, e);
        }
    }
}

// x = U^-1 L^-1 v, v = B z.  A channel's partitions are cut into segments of
// up to SN partitions, one work-group each, one lane per partition; a channel
// of at most 64 partitions is one segment.  With several segments a
// work-group also runs the PK partitions on either side of its own (halo):
// the forward carries need the pass-A end states of the PK partitions before
// them, and the backward carries need the PK partitions after the segment
// forward-solved.  Every value computed for an owned partition depends on
// these partitions only, so the segmentation does not change a single bit of
// the result.  Requires SN + 2 PK <= 64, or one segment.  ROLE is the RhsKind
// of the operator.
//
// What bounds it is latency: a lane's chain is 24 rows, four times, and the
// table rows (24 x P+1 units of 16 bytes for each of 64 partitions, 196 KB)
// neither fit the registers nor, with the buffers, the LDS.  On the small
// grids (STAGED: one work-group per compute unit) a work-group therefore has
// kWavesStaged waves.  Wave 0 runs the passes; at the start it loads the first
// block of rows into registers and 12 rows into LDS, where all four passes
// find them, and the remaining rows come from L2 a block ahead (Blocks).
// Meanwhile the helper waves fetch z, form v = B z (FUSE), and hold the
// transfer matrices, with which they run the carries.  Larger grids run one
// wave per work-group, several per compute unit, which hide each other's
// loads.
// Measured per launch, R, D, free and mask solves (with, in
// brackets, four waves that shared the passes' loads through LDS): 27.0 / 25.2 /
// 28.9 / 19.3 us at N = 3000 with 81 channels (32.2 / 27.6 / 33.8 / 22.8).  Of the
// 55 k cycles of a symmetric solve the passes take 27 k (two thirds of it the
// issue of their own arithmetic), the
// carries 7 k and the loads with the right-hand side 20 k.
//
// FUSE (STAGED): src is the state z and the work-group forms v = B z itself
// (the RhsKind ROLE with the bands of ra, the same arithmetic as k_rhs /
// k_rhs_shared) from the staged rows and P rows on either side of z in LDS;
// other work-groups read z rows this one owns, so src and zout may not
// overlap.  Without FUSE, src is v.
template <class TF, int P>
struct StageLds {
    // z rows of a fused right-hand side, then the carry's states (two
    // buffers) and the scrap rows of the passes that keep their input
    static constexpr int NZ = kPM * kLane + 2 * P;
    static constexpr int scrap = 2 * P * kSt;
    static constexpr int sz = NZ > scrap + kLane * Blocks<TF, P>::RB ? NZ : scrap + kLane * Blocks<TF, P>::RB;
    static constexpr int bytes =
        16 * (sz + kRowSlots + P * kSt + Blocks<TF, P>::LR * Blocks<TF, P>::UT * kLane);
    static_assert(bytes <= 160 * 1024, "LDS budget");
};

template <class TF, int ROLE, bool STAGED, bool FUSE, int P>
__global__ __launch_bounds__(kLane * (STAGED ? kWavesStaged : 1)) void k_bsolve(
    const cplx* __restrict__ tab, const TF* __restrict__ trf, TabMap tm, const cplx* __restrict__ src,
    cplx* __restrict__ zout, Geom geo, int SN, int PK, RhsArgs ra) {
    static_assert(STAGED || !FUSE, "the fused right-hand side is built for the staged grids");
    using F = TabFmt<TF, P>;
    using B = Blocks<TF, P>;
    using S = StageLds<TF, P>;
    constexpr int NTH = kLane * (STAGED ? kWavesStaged : 1);  // threads of the work-group
    __shared__ lcplx sv[kRowSlots];                             // the rows v, y, x
    __shared__ lcplx sE[P * kSt];                               // end states (one wave: the carry's)
    // z rows [r0 - P, r0 + NZ - P) (FUSE; zero outside [0, N)); then carry states and scrap rows
    __shared__ lcplx sz[STAGED ? S::sz : kLane * B::RB];
    __shared__ lcplx sT[STAGED ? B::LR * B::UT * kLane : 1];    // staged table rows

    int ch = blockIdx.y, seg = blockIdx.x;
    if (tm.order) {
        const int o = tm.order[blockIdx.y * gridDim.x + blockIdx.x];
        ch = o >> 8;
        seg = o & 255;
    }
    const int N = geo.N, NP = geo.P;
    const int k0 = seg * SN, k1 = min(NP, k0 + SN);         // owned partitions [k0, k1)
    const int ga = max(0, k0 - PK), gb = min(NP, k1 + PK);  // staged partitions [ga, gb)
    const int n = gb - ga;
    const int tid = threadIdx.x, ln = tid & (kLane - 1);
    const int w = STAGED ? __builtin_amdgcn_readfirstlane(tid / kLane) : 0;
    // this lane's partition; lanes past the staged ones repeat the last (their
    // rows and states are not used)
    const int g = min(ga + ln, gb - 1);
    const int tabid = table_of(tm, ch);
    const bool cj = conj_of(tm, ch);
    const int r0 = ga * kPM;  // first staged row
    const int nrow = n * kPM;
    const int nv = min(nrow, N - r0);  // staged rows below N
    const cplx* T = tab + (int64_t)tabid * F::units(geo);
    const unsigned off = part_off<TF, P>(g);
    const TF* TR = trf + (int64_t)tabid * F::trf_elems(geo);
    const unsigned toff = trf_off<TF, P>(g);
    const cplx* Tb = T + F::boff * kLane;                                   // backward units
    const cplx* Tb0 = Tb + (int64_t)(B::NB - 1) * B::RB * B::UT * kLane;    // their first block
    lcplx* rows = sv + row_slot(0, ln);

    if (w == 0) {
        BlockRegs<TF, P> c;
        cplx h[P];
        const lcplx* sL = sT + ln;
        lcplx* scrap = sz + (STAGED ? S::scrap : 0) + ln * B::RB;
        if constexpr (STAGED) {
            block_g<TF, P, F::UF>(c, T, off);
            // rows of blocks [LB0, LB1): straight into LDS, unit by unit
            const cplx* Ts = T + (int64_t)B::LB0 * B::RB * B::UT * kLane;
#pragma unroll 1
            for (int i = 0; i < B::LR; ++i)
#pragma unroll
                for (int u = 0; u < B::UT; ++u) {
                    const int d = F::SYM || u < B::UF ? i * B::UF + u : (B::LR + i) * B::UF + u - B::UF;
                    lds_load16((const cplx*)((const char*)(Ts + (i * B::UT + u) * kLane) + off), sT + d * kLane);
                }
            if (FUSE) __syncthreads();  // z in LDS
            __syncthreads();            // v in LDS
            lds_load_wait();
            // the states' zero columns (the z rows they replace are done with)
            if (ln < 2 * P) sz[ln * kSt + kLane] = lcplx{0.0, 0.0};
            if (ln < P) sE[ln * kSt + kLane] = lcplx{0.0, 0.0};
        } else {
            constexpr int KB = 8;  // rows fetched together
            const cplx* vi = src + (int64_t)ch * N + r0;
#pragma unroll 1
            for (int k = 0; k < kPM; k += KB) {
                cplx vr[KB];
#pragma unroll
                for (int j = 0; j < KB; ++j) vr[j] = cj_if(cj, vi[min(tid + (k + j) * NTH, nv - 1)]);
#pragma unroll
                for (int j = 0; j < KB; ++j) {
                    const int i = tid + (k + j) * NTH;
                    if (i < nrow) sv[row_slot(i % kPM, i / kPM)] = lc(i < nv ? vr[j] : cplx{0.0, 0.0});
                }
            }
            block_g<TF, P, F::UF>(c, T, off);
            if (ln < P) sE[ln * kSt + kLane] = lcplx{0.0, 0.0};
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < P; ++j) h[j] = {0.0, 0.0};
        // forward: pass A from the zero state, carry, pass B
#pragma unroll 1
        for (int pass = 0;; ++pass) {
            fwd_pass<TF, P, STAGED>(c, T, off, sL, rows, pass ? rows : scrap, pass ? B::RB : 0, h, pass ? Tb0 : T);
            if (pass) break;
            if constexpr (STAGED) {
#pragma unroll
                for (int j = 0; j < P; ++j) sE[j * kSt + ln] = lc(h[j]);
                for (int k = 0; k < PK; ++k) __syncthreads();
                const lcplx* s = carried<P>(sE, sz, PK) + neighbour(ln, n, 0);
#pragma unroll
                for (int j = 0; j < P; ++j) h[j] = s[j * kSt];
            } else {
                TF t[P][P];
                // loaded here: left to the compiler it is loaded in the pass, in every
                // block again, and fills the registers (608 / 882 / 1020 channels of
                // N = 1200, R part: 53.6 / 70.2 / 75.5 us, here 47.9 / 62.2 / 67.8)
                const TF* Tq = TR;
                asm volatile("" : "+s"(Tq));
#pragma unroll
                for (int r = 0; r < P; ++r)
#pragma unroll
                    for (int q = 0; q < P; ++q) t[r][q] = trf_at<TF, P>(Tq, toff, 0, r, q);
                carry1<TF, P>(t, sE, ln, n, 0, PK, h);
            }
        }
        if constexpr (STAGED && !F::SYM) sL += B::LR * B::UF * kLane;
#pragma unroll
        for (int j = 0; j < P; ++j) h[j] = {0.0, 0.0};
#pragma unroll 1
        for (int pass = 0;; ++pass) {
            bwd_pass<TF, P, STAGED>(c, Tb, off, sL, rows, pass ? rows : scrap, pass ? B::RB : 0, h, Tb0);
            if (pass) break;
            if constexpr (STAGED) {
#pragma unroll
                for (int j = 0; j < P; ++j) sE[j * kSt + ln] = lc(h[j]);
                for (int k = 0; k < PK; ++k) __syncthreads();
                const lcplx* s = carried<P>(sE, sz, PK) + neighbour(ln, n, 1);
#pragma unroll
                for (int j = 0; j < P; ++j) h[j] = s[j * kSt];
            } else {
                TF t[P][P];
                const TF* Tq = TR;
                asm volatile("" : "+s"(Tq));  // loaded here: kept from the forward carry it would fill the registers
#pragma unroll
                for (int r = 0; r < P; ++r)
#pragma unroll
                    for (int q = 0; q < P; ++q) t[r][q] = trf_at<TF, P>(Tq, toff, 1, r, q);
                carry1<TF, P>(t, sE, ln, n, 1, PK, h);
            }
        }
    } else {
        constexpr int HT = kLane * kHelp, NR = kPM * kLane;  // helper threads, rows
        constexpr int KH = (NR + HT - 1) / HT;               // rows per thread
        const int ht = tid - kLane, hw = w - 1;
        TF t[trf_rows(P)][P];
        if constexpr (FUSE) {
            using Row = std::conditional_t<ROLE == RHS_CBAND, CBandRow<P>, SBandRow<ROLE, P>>;
            constexpr int KZ = (S::NZ + HT - 1) / HT;
            const cplx* zc = src + (int64_t)ch * N;
            const int zlo = r0 - P;
            cplx zr[KZ];
#pragma unroll
            for (int k = 0; k < KZ; ++k) zr[k] = cj_if(cj, zc[min(max(zlo + ht + k * HT, 0), N - 1)]);
            // (two matrix rows beside two band rows would not fit the registers)
            if constexpr (trf_rows(P) == 1) carry_load<TF, P>(t, TR, toff, 0, hw);
            auto row_at = [&](int k) { return min(r0 + min(ht + k * HT, NR - 1), N - 1); };
            auto band = [&](Row& b, int k) {
                if constexpr (ROLE == RHS_CBAND) b.load(ra.cband + (int64_t)tabid * (P + 1) * N, row_at(k), N);
                else b.load(ra, row_at(k), N);
            };
            // staged row i is channel row r0 + i, its z_{r0+i+d} sits at
            // sz[i + P + d]; a conjugate channel forms its table's
            // right-hand side (scalar -e)
            const double e0 = ROLE == RHS_SX_SYM || ROLE == RHS_SX_ASY ? ra.eig[ch] * ra.ifdt : 0.0;
            const double e = cj ? -e0 : e0;
            auto form = [&](const Row& b, int k) {
                const int i = min(ht + k * HT, NR - 1);  // (a row past the last repeats the last)
                cplx v;
                auto zat = [&](int d) -> cplx { return sz[i + P + d]; };
                if constexpr (ROLE == RHS_CBAND) v = b.apply(zat, row_at(k));
                else v = b.apply(zat, e);
                // rows from N on are padding: v = 0
                if (i < nrow) sv[row_slot(i % kPM, i / kPM)] = lc(i < nv ? v : cplx{0.0, 0.0});
            };
            // band entries a row ahead of the products
            Row b0, b1;
            band(b0, 0);
#pragma unroll
            for (int k = 0; k < KZ; ++k) {
                const int j = ht + k * HT, row = zlo + j;
                if (j < S::NZ) sz[j] = lc(row >= 0 && row < N ? zr[k] : cplx{0.0, 0.0});
            }
            __syncthreads();
#pragma unroll 1
            for (int k = 0; k < KH; k += 2) {
                band(b1, k + 1);
                __builtin_amdgcn_sched_barrier(0);
                form(b0, k);
                band(b0, min(k + 2, KH - 1));
                __builtin_amdgcn_sched_barrier(0);
                form(b1, k + 1);
            }
            if constexpr (trf_rows(P) > 1) carry_load<TF, P>(t, TR, toff, 0, hw);
        } else {
            const cplx* vi = src + (int64_t)ch * N + r0;
            cplx vr[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) vr[k] = cj_if(cj, vi[min(ht + k * HT, nv - 1)]);
            carry_load<TF, P>(t, TR, toff, 0, hw);
#pragma unroll
            for (int k = 0; k < KH; ++k) {
                const int i = ht + k * HT;
                if (i < nrow) sv[row_slot(i % kPM, i / kPM)] = lc(i < nv ? vr[k] : cplx{0.0, 0.0});
            }
        }
        __syncthreads();  // v in LDS
#pragma unroll 1
        for (int dir = 0;; ++dir) {
            __syncthreads();  // end states
            carry8<TF, P>(t, sE, sz, ln, n, dir, PK, hw);
            if (dir) break;
            carry_load<TF, P>(t, TR, toff, 1, hw);
        }
    }
    __syncthreads();
    const int i0 = (k0 - ga) * kPM, i1 = min((k1 - ga) * kPM, nv);
    cplx* xo = zout + (int64_t)ch * N + r0;
#pragma unroll 6
    for (int i = i0 + tid; i < i1; i += NTH) xo[i] = cj_if(cj, sv[row_slot(i % kPM, i / kPM)]);
}

// The same solve, bit for bit, with eight lanes per partition, for channels of
// at most kSplitParts partitions and for longer ones on small grids, where
// k_bsolve's waves would leave lanes or compute units idle.  Lane l owns rows l,
// l + 8 and l + 16 of its partition.  Going down, the row's value is broadcast
// to the eight (two DPP moves per double) and each lane subtracts its multiple
// from the row it gathers next: P products per row in one instruction each, and
// the chain of a row is the sum with its right-hand side, a broadcast and two
// FMAs.  Going up is the same from the last row, which begin with their values,
// with the rows' own coefficients.  The state a partition hands down is what the eight
// lanes have gathered for the first rows of the next one.  A lane's 24
// coefficients per direction stay in registers for both passes, its rows too:
// LDS holds the rows of z for the right-hand side, P rows on either side, and
// the states of the carries, which each lane runs for its own entry (row l of
// the transfer matrix).
//
// A pass takes 1.6 k cycles (k_bsolve: 6.5 k), so what bounds it is the loads:
// every table entry twice, the band entries of three rows per lane.  More
// partitions to a work-group would wait for them as long as k_bsolve does (64 at
// N = 1500: no gain), and so would two work-groups to a compute unit; fewer wait
// less (split_grid).  R, D, free and mask solves of 6 channels of N = 240: 13.2 /
// 11.4 / 12.7 / 9.7 us (k_bsolve 21.6 / 18.0 / 21.4 / 17.0).  At 32 partitions,
// uncut, 31 channels step by step 5.3 -> 4.3 ms, 2400 batched ones 36.0 -> 31.1.
// A step of longer channels, k_bsolve before: 31 of N = 1000 155 -> 102 us, 41 of
// N = 1500 167 -> 118, 51 of N = 2000 175 -> 140, 30 of N = 3000 170 -> 132.
//
// FUSE: as k_bsolve's; with one segment src and zout may be the same.
constexpr int kSplit = 8;                     // lanes per partition
constexpr int kSplitParts = 32;               // partitions up to which they are used
constexpr int64_t kSplitGrid = 256;           // work-groups of a cut grid, one per compute unit
constexpr int kOwn = kPM / kSplit;            // rows per lane
constexpr int kSt8 = kSplit + 1;              // a state's entries in LDS, odd for the banks
static_assert(kPM % kSplit == 0 && kSplit == 8, "lane layout");

template <int L>
__device__ inline double bcast8(double v) {  // lane L of each eight
    const long long b = __double_as_longlong(v);
    const long long a = __builtin_amdgcn_mov_dpp(b, 0x150 + L, 0xf, 0xf, true);
    return __longlong_as_double(__builtin_amdgcn_update_dpp(a, b, 0x158 + L, 0xf, 0xc, false));
}
template <int L>
__device__ inline cplx bcast8(cplx v) { return {bcast8<L>(v.re), bcast8<L>(v.im)}; }
__device__ inline cplx pick(bool c, cplx a, cplx b) { return {c ? a.re : b.re, c ? a.im : b.im}; }
// keeps a value where it is computed: put off to its use, it would keep its
// operands alive until then
__device__ inline void keep(cplx& v) { asm volatile("" : "+v"(v.re), "+v"(v.im)); }

// A lane's coefficients.  ld: byte offset of coefficient k = 1..P of row `row`
// (relative to the table's partition column), element P the diagonal
template <class TF, int P>
struct LaneTab {
    using F = TabFmt<TF, P>;
    static constexpr unsigned kUnit = kLane * 16u, kRow = F::row * kUnit;
    __device__ static unsigned elem(int e) {  // element e = 0..P of a row
        if constexpr (F::SYM) return (unsigned)e * kUnit;
        else return (unsigned)(e >> 1) * kUnit + (unsigned)(e & 1) * 8u;
    }
    __device__ static TF at(const char* base, unsigned off) { return *(const TF*)(base + off); }
};

// rows down through the partition: z the own rows' right-hand sides, each added
// when its row is done (fwd_row), acc what the partition above contributes (in)
// and what this one does to the next (out), y the own rows
template <int P>
__device__ inline void rows_down(const cplx (&C)[kPM], const cplx (&z)[kOwn], cplx (&y)[kOwn], cplx& acc, int l) {
    each(std::make_integer_sequence<int, kPM>{}, [&](auto sc) {
        constexpr int s = decltype(sc)::value, t = s / kSplit, r = s % kSplit;
        const cplx w = {z[t].re + acc.re, z[t].im + acc.im};
        const cplx x = bcast8<r>(w);
        y[t] = pick(l == r, w, y[t]);
        keep(y[t]);
        acc = tmsub(pick(l == r, cplx{0.0, 0.0}, acc), C[s], x);
    });
}
// rows up; acc: the last eight's y less what the partition below contributes
template <int P>
__device__ inline void rows_up(const cplx (&C)[kPM], const cplx (&y)[kOwn], cplx (&x)[kOwn], cplx acc, int l) {
    each(std::make_integer_sequence<int, kPM>{}, [&](auto sc) {
        constexpr int s = kPM - 1 - decltype(sc)::value, t = s / kSplit, r = s % kSplit;
        const cplx v = bcast8<r>(acc);
        x[t] = pick(l == r, acc, x[t]);
        keep(x[t]);
        if constexpr (s > 0) {
            if constexpr (t > 0) acc = pick(l == r, y[t - 1], acc);
            acc = tmsub(acc, C[s], v);
        }
    });
}

// The same for real tables, whose coefficients leave room for two of each:
// C[s] where lane l still gathers its row of this eight (l past row s), B[s]
// where it gathers the next eight's, zero elsewhere.  Then no value is picked:
// two products for eight moves (a step of 6 channels of N = 240 83 -> 80 us).
template <int P>
__device__ inline void rows_down_r(const double (&C)[kPM], const double (&B)[kPM], const double (&dg)[kOwn],
                                   const cplx (&z)[kOwn], cplx (&y)[kOwn], cplx& acc) {
    cplx a[kOwn + 1];
    a[0] = acc;
#pragma unroll
    for (int t = 1; t <= kOwn; ++t) a[t] = {0.0, 0.0};
    each(std::make_integer_sequence<int, kPM>{}, [&](auto sc) {
        constexpr int s = decltype(sc)::value, t = s / kSplit, r = s % kSplit;
        const cplx x = bcast8<r>(cplx{dg[t] * (z[t].re + a[t].re), dg[t] * (z[t].im + a[t].im)});
        if constexpr (r < kSplit - 1) a[t] = tmsub(a[t], C[s], x);
        if constexpr (r > 0 || P == 8) a[t + 1] = tmsub(a[t + 1], B[s], x);
    });
#pragma unroll
    for (int t = 0; t < kOwn; ++t) y[t] = {dg[t] * (z[t].re + a[t].re), dg[t] * (z[t].im + a[t].im)};
    acc = a[kOwn];
}
template <int P>
__device__ inline void rows_up_r(const double (&C)[kPM], const double (&B)[kPM], const cplx (&y)[kOwn],
                                 cplx (&x)[kOwn], cplx acc) {
    x[kOwn - 1] = acc;
#pragma unroll
    for (int t = 0; t + 1 < kOwn; ++t) x[t] = y[t];
    each(std::make_integer_sequence<int, kPM>{}, [&](auto sc) {
        constexpr int s = kPM - 1 - decltype(sc)::value, t = s / kSplit, r = s % kSplit;
        const cplx v = bcast8<r>(x[t]);
        if constexpr (r > 0) x[t] = tmsub(x[t], C[s], v);
        if constexpr (t > 0 && (r < kSplit - 1 || P == 8)) x[t > 0 ? t - 1 : 0] = tmsub(x[t > 0 ? t - 1 : 0], B[s], v);
    });
}

// The incoming states from the pass-A end states e: s_g <- e_g + T_g s_{g-1}
// (g+1 backward), PK - 1 times from s = e, so that s_{g-1} holds the PK
// partitions before g, the same sums as Horner's rule over them.  Entry l of
// slot q at q * kSt8 + l; slot nb is the neighbour's, or the zero slot.  Returns
// the neighbour's incoming state.
// (par: which buffer comes first, so that a direction's first is not the
// other's last, which lanes may still be reading)
template <class TF, int P>
__device__ inline const lcplx* carry(lcplx (*sS)[(kSplitParts + 1) * kSt8], const TF (&t)[P], cplx e, int own, int nb, int PK,
                                     int par) {
    cplx a = e;
#pragma unroll 1
    for (int k = 1;; ++k) {
        lcplx* buf = sS[(k + par) & 1];
        buf[own] = lc(a);
        __syncthreads();
        if (k == PK) return buf + nb * kSt8;
        cplx in[P];
#pragma unroll
        for (int c = 0; c < P; ++c) in[c] = buf[nb * kSt8 + c];
        a = e;
#pragma unroll
        for (int c = 0; c < P; ++c) a = tmac(a, t[c], in[c]);
    }
}

// row r of the direction's matrix
template <class TF, int P>
__device__ inline void trf_row(TF (&t)[P], const TF* T, unsigned off, int dir, int r) {
    constexpr bool SYM = TabFmt<TF, P>::SYM;
    const bool tr = SYM && dir;
    const unsigned o = off + (unsigned)((SYM ? 0 : dir * P * P) + (tr ? r : r * P)) * kLane * (unsigned)sizeof(TF);
#pragma unroll
    for (int c = 0; c < P; ++c) t[c] = *(const TF*)((const char*)(T + (tr ? c * P : c) * kLane) + o);
}

template <class TF, int ROLE, bool FUSE, int P>
__global__ __launch_bounds__(kSplitParts * kSplit) void k_bsolve8(const cplx* __restrict__ tab, const TF* __restrict__ trf,
                                                           TabMap tm, const cplx* __restrict__ src,
                                                           cplx* __restrict__ zout, Geom geo, int SN, int SX,
                                                           int PK, RhsArgs ra) {
    using F = TabFmt<TF, P>;
    using LT = LaneTab<TF, P>;
    constexpr bool SYM = F::SYM;
    constexpr int KZ = 4;  // staged rows per thread: 24 per eight threads, and 2 P
    __shared__ lcplx sz[FUSE ? kPM * kSplitParts + 2 * P : 1];  // z rows [r0 - P, r0 + nrow + P), zero outside [0, N)
    __shared__ lcplx sS[2][(kSplitParts + 1) * kSt8];            // states

    int ch = blockIdx.y, seg = blockIdx.x;
    if (tm.order) {
        const int o = tm.order[blockIdx.y * gridDim.x + blockIdx.x];
        ch = o >> 8;
        seg = o & 255;
    }
    const int N = geo.N, NP = geo.P;
    // owned partitions [k0, k1): SN, the first segment's SX more, the last one's what is left
    const int k0 = seg ? SX + seg * SN : 0, k1 = seg == (int)gridDim.x - 1 ? NP : SX + (seg + 1) * SN;
    const int ga = max(0, k0 - PK), gb = min(NP, k1 + PK);  // staged partitions [ga, gb)
    const int n = gb - ga;
    const int tid = threadIdx.x, q = tid / kSplit, l = tid % kSplit;
    // this lane's partition; slots past the staged ones repeat the last (their
    // rows and states are not used)
    const int g = min(ga + q, gb - 1);
    const int tabid = table_of(tm, ch);
    const bool cj = conj_of(tm, ch);
    const int r0 = ga * kPM;  // first staged row
    const int i0 = g * kPM + l;
    const char* T = (const char*)(tab + (int64_t)tabid * F::units(geo));
    const unsigned off = part_off<TF, P>(g);
    const TF* TR = trf + (int64_t)tabid * F::trf_elems(geo);
    const unsigned toff = trf_off<TF, P>(g);
    const int own = q * kSt8 + l, lp = min(l, P - 1);

    if (tid < 2 * kSt8) sS[tid / kSt8][kSplitParts * kSt8 + tid % kSt8] = lcplx{0.0, 0.0};
    // requests: z, the first band row, the forward coefficients
    using Row = std::conditional_t<ROLE == RHS_CBAND, CBandRow<P>, SBandRow<ROLE, P>>;
    Row band;
    auto load_band = [&](int t) {
        const int i = min(i0 + kSplit * t, N - 1);
        if constexpr (ROLE == RHS_CBAND) band.load(ra.cband + (int64_t)tabid * (P + 1) * N, i, N);
        else band.load(ra, i, N);
    };
    cplx z[kOwn], zr[FUSE ? KZ : 1];
    if constexpr (FUSE) {
        const cplx* zc = src + (int64_t)ch * N;
#pragma unroll
        for (int k = 0; k < KZ; ++k) zr[k] = zc[min(max(r0 - P + tid + k * (int)blockDim.x, 0), N - 1)];
        load_band(0);
    } else {
#pragma unroll
        for (int t = 0; t < kOwn; ++t) z[t] = src[(int64_t)ch * N + min(i0 + kSplit * t, N - 1)];
    }
    TF C[kPM], dg[kOwn], tr[P];
    auto load_down = [&](int t) {
#pragma unroll
        for (int r = 0; r < kSplit; ++r)
            C[t * kSplit + r] = LT::at(T + t * kSplit * LT::kRow, off + r * LT::kRow + LT::elem((l - r - 1) & 7));
        dg[t] = LT::at(T + t * kSplit * LT::kRow, off + l * LT::kRow + LT::elem(P));
    };
    // (the right-hand side's operands leave room for two thirds of them)
    constexpr int T0 = FUSE ? 2 : kOwn;
#pragma unroll
    for (int t = 0; t < T0; ++t) load_down(t);
    if constexpr (FUSE) {
        const int nz = n * kPM + 2 * P, zlo = r0 - P;
#pragma unroll
        for (int k = 0; k < KZ; ++k) {
            const int j = tid + k * blockDim.x, row = zlo + j;
            if (j < nz) sz[j] = lc(row >= 0 && row < N ? cj_if(cj, zr[k]) : cplx{0.0, 0.0});
        }
        __syncthreads();
        // staged row i is channel row r0 + i, its z_{r0+i+d} sits at sz[i + P +
        // d]; a conjugate channel forms its table's right-hand side (scalar -e)
        const double e0 = ROLE == RHS_SX_SYM || ROLE == RHS_SX_ASY ? ra.eig[ch] * ra.ifdt : 0.0;
        const double e = cj ? -e0 : e0;
#pragma unroll 1
        for (int t = 0; t < kOwn; ++t) {
            const int i = i0 + kSplit * t;
            const lcplx* zs = sz + (i - r0 + P);
            cplx v;
            // four rows of z at a time: all fifteen would leave too few registers for the coefficients
            auto zat = [&](int d) -> cplx {
                if (d % 4 == 0) __builtin_amdgcn_sched_barrier(0);
                return zs[d];
            };
            if constexpr (ROLE == RHS_CBAND) v = band.apply(zat, min(i, N - 1));
            else v = band.apply(zat, e);
            if (i >= N) v = cplx{0.0, 0.0};  // padding
#pragma unroll
            for (int k = 0; k + 1 < kOwn; ++k) z[k] = z[k + 1];
            z[kOwn - 1] = v;
            keep(v);  // (before the next row's entries are requested)
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1 < kOwn) load_band(t + 1);
        }
    } else {
#pragma unroll
        for (int t = 0; t < kOwn; ++t) z[t] = i0 + kSplit * t < N ? cj_if(cj, z[t]) : cplx{0.0, 0.0};
    }
#pragma unroll
    for (int t = T0; t < kOwn; ++t) load_down(t);
    trf_row<TF, P>(tr, TR, toff, 0, lp);

    // Coefficients of the way up: row 8 t + r reaches lane l's row of its eight
    // or of the eight above (the first rows' wrap around: the partition's last
    // eight, which the partition below reaches).  The last rows' are requested
    // here (a real table's all), the others once the way down has left room.
    TF D[kPM];
    auto load_up = [&](int t) {
#pragma unroll
        for (int r = kSplit - 1; r >= 0; --r) {
            const bool same = P == 7 ? l <= r : l < r;
            const unsigned o = off + (unsigned)F::boff * LT::kUnit + LT::elem((r - l - 1) & 7);
            const int row = t ? (same ? l + kSplit : l) : (same ? l : kPM - kSplit + l);
            D[t * kSplit + r] = LT::at(T + (t ? t - 1 : 0) * kSplit * LT::kRow, o + (unsigned)row * LT::kRow);
        }
    };
    constexpr int T1 = SYM ? (P == 7 ? 2 : kOwn) : 0;
#pragma unroll
    for (int t = kOwn - 1; t >= T1; --t) load_up(t);
    // down: pass A from the zero state, carry, pass B
    TF B[SYM ? 1 : kPM];
    if constexpr (!SYM) {
#pragma unroll
        for (int s = 0; s < kPM; ++s) {
            B[s] = (P == 8 ? l <= s % kSplit : l < s % kSplit) ? C[s] : 0.0;
            C[s] = l > s % kSplit ? C[s] : 0.0;
        }
    } else if constexpr (P == 7) {
#pragma unroll
        for (int s = 0; s < kPM; ++s) C[s] = pick(l == s % kSplit, tzero(TF{}), C[s]);
    }
    cplx y[kOwn], acc = {0.0, 0.0};
#pragma unroll
    for (int t = 0; t < kOwn; ++t) y[t] = acc;
#pragma unroll 1
    for (int pass = 0;; ++pass) {
        if constexpr (SYM) rows_down<P>(C, z, y, acc, l);
        else rows_down_r<P>(C, B, dg, z, y, acc);
        if (pass) break;
        const lcplx* in = carry<TF, P>(sS, tr, acc, own, q > 0 && q < n ? q - 1 : kSplitParts, PK, 0);
        acc = l < P ? (cplx)in[l] : cplx{0.0, 0.0};
    }
    // up
#pragma unroll
    for (int t = T1 - 1; t >= 0; --t) load_up(t);
    trf_row<TF, P>(tr, TR, toff, 1, lp);
#pragma unroll
    for (int t = 0; t < kOwn; ++t) {
        if constexpr (SYM) {
            y[t] = tmulf(dg[t], y[t]);
        } else {
            const TF d = LT::at(T + t * kSplit * LT::kRow, off + (unsigned)F::boff * LT::kUnit + l * LT::kRow + LT::elem(P));
            y[t] = {d * y[t].re, d * y[t].im};
        }
    }
    cplx x[kOwn];
    if constexpr (!SYM) {
#pragma unroll
        for (int s = kPM - 1; s >= 0; --s) {
            B[s] = (P == 8 ? l >= s % kSplit : l > s % kSplit) ? D[s] : 0.0;
            D[s] = l < s % kSplit ? D[s] : 0.0;
        }
    } else if constexpr (P == 7) {
#pragma unroll
        for (int s = kPM - 1; s >= 0; --s) D[s] = pick(l == s % kSplit, tzero(TF{}), D[s]);
    }
#pragma unroll
    for (int t = 0; t < kOwn; ++t) x[t] = {0.0, 0.0};
    acc = y[kOwn - 1];
#pragma unroll 1
    for (int pass = 0;; ++pass) {
        if constexpr (SYM) rows_up<P>(D, y, x, acc, l);
        else rows_up_r<P>(D, B, y, x, acc);
        if (pass) break;
        const lcplx* in = carry<TF, P>(sS, tr, x[0], own, q + 1 < n ? q + 1 : kSplitParts, PK, PK);
        // the first P rows of the partition below, seen from this one's last eight
#pragma unroll
        for (int i = P - 1; i >= 0; --i) {
            const bool on = P == 7 ? l > i : l >= i;
            if constexpr (SYM) acc = tmsub(acc, pick(on, D[i], tzero(TF{})), (cplx)in[i]);
            else acc = tmsub(acc, B[i], (cplx)in[i]);
        }
    }
    cplx* xo = zout + (int64_t)ch * N;
    if (q >= k0 - ga && q < k1 - ga)
#pragma unroll
        for (int t = 0; t < kOwn; ++t)
            if (i0 + kSplit * t < N) xo[i0 + kSplit * t] = cj_if(cj, x[t]);
}

// Sequential solve x = U^-1 L^-1 v over all N rows, one lane per channel:
// the fallback for carries deeper than kPKMax partitions (exact for any
// operator the tables hold).  Table rows are fetched in blocks of RB rows,
// every load of a block issued before its first use and none under a branch
// (rows from N on repeat the last and are left out); zout holds y between
// the two passes.
template <class TF, int P>
__global__ __launch_bounds__(64) void k_seqsolve(const cplx* __restrict__ tab, TabMap tm, const cplx* __restrict__ vin,
                                                 cplx* __restrict__ zout, Geom geo, int nch) {
    using F = TabFmt<TF, P>;
    constexpr int RB = 6;
    const int ch = blockIdx.x * 64 + threadIdx.x;
    if (ch >= nch) return;
    const int N = geo.N;
    const cplx* T0 = tab + (int64_t)table_of(tm, ch) * F::units(geo);
    const bool cj = conj_of(tm, ch);
    const cplx* v = vin + (int64_t)ch * N;
    cplx* x = zout + (int64_t)ch * N;
    cplx h[P];
#pragma unroll
    for (int j = 0; j < P; ++j) h[j] = {0.0, 0.0};
    for (int i0 = 0; i0 < N; i0 += RB) {
        cplx c[RB][F::UF], vr[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int i = min(i0 + b, N - 1);
            row_g<TF, P, F::UF>(c[b], T0, part_off<TF, P>(i / kPM), i % kPM);
            vr[b] = cj_if(cj, v[i]);
        }
#pragma unroll
        for (int b = 0; b < RB; ++b)
            if (i0 + b < N) x[i0 + b] = fwd_row<TF, P>(c[b], vr[b], h);
    }
#pragma unroll
    for (int j = 0; j < P; ++j) h[j] = {0.0, 0.0};
    for (int i1 = N - 1; i1 >= 0; i1 -= RB) {
        cplx c[RB][F::UF], yr[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int i = max(i1 - b, 0);
            row_g<TF, P, F::UF>(c[b], T0 + F::boff * kLane, part_off<TF, P>(i / kPM), i % kPM);
            yr[b] = x[i];
        }
#pragma unroll
        for (int b = 0; b < RB; ++b)
            if (i1 - b >= 0) x[i1 - b] = cj_if(cj, bwd_row<TF, P>(c[b], yr[b], h));
    }
}

// ---------------------------------------------------------------------------
// Transfer matrices: one lane per (table, partition), the unit responses of
// the state through the partition's rows, NC at a time (as many as the
// registers hold beside the rows), the groups of columns - and, of real LU
// tables, the two directions - in work-groups of their own.  A symmetric
// table's backward matrix is the transpose of the forward one and is not
// stored.  Rows are loaded in blocks of RB ahead of their products.
template <class TF, int P>
constexpr int trf_cols() { return TabFmt<TF, P>::SYM ? 4 : P; }
template <class TF, int P>
constexpr int trf_groups() { return TabFmt<TF, P>::SYM ? (P + trf_cols<TF, P>() - 1) / trf_cols<TF, P>() : 2; }

__device__ inline double tsub(double a, double t, double x) { return fma(-t, x, a); }
__device__ inline cplx tsub(cplx a, cplx t, cplx x) { return tmsub(a, t, x); }

template <class TF, int P>
__device__ inline void transfer_cols(const cplx* __restrict__ tab, TF* __restrict__ trf, Geom geo, int64_t t) {
    using F = TabFmt<TF, P>;
    constexpr int NC = trf_cols<TF, P>(), RB = 4;
    const int grp = blockIdx.y % trf_groups<TF, P>();
    const int g = blockIdx.y / trf_groups<TF, P>() * kLane + threadIdx.x;
    if (g >= geo.P) return;
    const int dir = F::SYM ? 0 : grp, c0 = F::SYM ? grp * NC : 0;
    const cplx* T0 = tab + t * F::units(geo) + (dir ? F::boff * kLane : 0);
    const unsigned off = part_off<TF, P>(g);
    TF* out = trf + t * F::trf_elems(geo) + (int64_t)(g >> 6) * (F::SYM ? 1 : 2) * P * P * kLane +
              (int64_t)dir * P * P * kLane + (g & 63);
    TF H[P][NC];  // H[q][c]: state entry q of the response to unit vector c0 + c
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c) H[q][c] = q == c0 + c ? tone(TF{}) : tzero(TF{});
#pragma unroll 1
    for (int s0 = 0; s0 < kPM; s0 += RB) {
        cplx e[RB][F::UF];
#pragma unroll
        for (int b = 0; b < RB; ++b) row_g<TF, P, F::SYM ? P : F::UF>(e[b], T0, off, dir ? kPM - 1 - s0 - b : s0 + b);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            if (!F::SYM && dir) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    TF x = tzero(TF{});
#pragma unroll
                    for (int k = P; k >= 1; --k) x = tsub(x, F::coef(e[b], k), H[k - 1][c]);
#pragma unroll
                    for (int q = P - 1; q > 0; --q) H[q][c] = H[q - 1][c];
                    H[0][c] = x;
                }
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    TF y = H[0][c];
                    if constexpr (!F::SYM) y = F::diag(e[b]) * y;
#pragma unroll
                    for (int k = 1; k < P; ++k) H[k - 1][c] = tsub(H[k][c], F::coef(e[b], k), y);
                    H[P - 1][c] = tsub(tzero(TF{}), F::coef(e[b], P), y);
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (c0 + c < P) out[(int64_t)(q * P + c0 + c) * kLane] = H[q][c];
}
template <class TF, int P>
__global__ __launch_bounds__(kLane) void k_transfer(const cplx* __restrict__ tab, TF* __restrict__ trf, Geom geo,
                                                    int64_t stride) {
    transfer_cols<TF, P>(tab, trf, geo, (int64_t)blockIdx.z * stride + blockIdx.x);
}

// ---------------------------------------------------------------------------
// complex symmetric tables from the lu_zsb factor (ed.h:208-289):
// f[i*ne] = D_i, f[i*ne+j] = L(i+j,i); one lane per (table, partition)
template <int P>
__global__ __launch_bounds__(kLane) void k_tab_ldlt(const cplx* __restrict__ lower, cplx* __restrict__ tab, Geom geo) {
    constexpr int R = P + 1, ne = P + 1;
    const int g = blockIdx.x * kLane + threadIdx.x;
    const int l = blockIdx.y;
    if (g >= geo.P) return;
    const int N = geo.N;
    const cplx* f = lower + (int64_t)l * N * ne;
    cplx* Tg = tab + (int64_t)l * geo.ctab_elems + part_col<cplx, P>(g);
    for (int s = 0; s < kPM; ++s) {
        const int i = g * kPM + s;
        cplx o[R];
        if (i >= N) {  // identity padding row
#pragma unroll
            for (int q = 0; q < P; ++q) o[q] = {0.0, 0.0};
            o[P] = {1.0, 0.0};
        } else {
#pragma unroll
            for (int k = 1; k <= P; ++k) o[k - 1] = i + k < N ? f[(int64_t)i * ne + k] : cplx{0.0, 0.0};
            o[P] = crecip(f[(int64_t)i * ne]);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) Tg[(int64_t)(s * R + q) * kLane] = o[q];
    }
}

// tables from chol(S) (ed.h:182-194): c[i*ne+j] = L(i+j,i)
template <int P>
__global__ __launch_bounds__(kLane) void k_tab_chol(const double* __restrict__ c, cplx* __restrict__ tab, Geom geo) {
    using F = TabFmt<double, P>;
    constexpr int ne = P + 1;
    const int g = blockIdx.x * kLane + threadIdx.x;
    if (g >= geo.P) return;
    const int N = geo.N;
    cplx* Tg = tab + part_col<double, P>(g);
    for (int s = 0; s < kPM; ++s) {
        const int i = g * kPM + s;
        double f[P], b[P], d = 1.0;  // identity padding rows
#pragma unroll
        for (int k = 0; k < P; ++k) f[k] = b[k] = 0.0;
        if (i < N) {
            d = 1.0 / c[(int64_t)i * ne];
#pragma unroll
            for (int k = 1; k <= P; ++k)
                if (i + k < N) {
                    f[k - 1] = c[(int64_t)i * ne + k];
                    b[k - 1] = f[k - 1] * d;
                }
        }
        put_real<P>(Tg + (int64_t)s * F::row * kLane, f, d);
        put_real<P>(Tg + (int64_t)(s * F::row + F::boff) * kLane, b, d);
    }
}

__global__ __launch_bounds__(256) void k_band_pair(const double* __restrict__ S, const double* __restrict__ X,
                                                   cplx* __restrict__ dst, int64_t total) {
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id < total) dst[id] = cplx{S[id], X[id]};
}

template <class T>
__global__ __launch_bounds__(256) void k_band_diag(const T* __restrict__ src, T* __restrict__ dst, int64_t total,
                                                   int N, int ne) {
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const int64_t b = id / ((int64_t)ne * N);
    const int64_t r = id % ((int64_t)ne * N);
    const int j = (int)(r / N), i = (int)(r % N);
    dst[id] = src[(b * N + i) * ne + j];
}

// ---------------------------------------------------------------------------
// LU of A = S + ifet X in the reference's elimination order
// (propagate.hpp:33-86), one lane per (time point, channel, partition).  A
// lane restarts the elimination `above` rows above its partition (as if the
// matrix began there) and writes the table rows of its own partition.
//
// The elimination is right-looking: the lane keeps the window of the Schur
// complement that row i touches (rows and columns i .. i+P) in registers; row
// r's entries sit in slot (r - start) mod RS, and the row loop is unrolled by
// the RS slots so that every slot index is a constant.  A symmetric
// matrix (S + i e X) needs the upper triangle only, P(P+1)/2 products per row
// where the row-by-row elimination forms P^2.  Column i + P of the band
// enters the window at step i; its {S, X} entries (launch_factor_bands) lie
// partition-interleaved, so that a wave's load is one contiguous run instead of
// 64 lines 24 rows apart, and the next column is loaded a whole step ahead.
// Few tables are bound by the chain of rows (reciprocal, scale, update of
// the next pivot: 31 channels of N = 1000 take 41 us, was 134) and are left to
// k_factor_row.  A batch is bound by the products and the table
// writes: 32 time points of N = 3000, 41 tables of S + i e X 167 us (was
// 434), 81 of S + e X 307 us (was 596).
//
// Both kernels start the same number of rows above a partition, whole rounds of
// either (8 rows; 12 and 8 for p = 8), so that a table's bits do not depend on
// how many are built together.
constexpr int restart_round(int p) { return p == 7 ? 8 : 24; }
static int restart_rows(int p, int restart) {
    const int r = restart_round(p);
    return ((restart > 0 ? restart : kRestart) + r - 1) / r * r;
}

template <int SYM>
struct FactorTypes;
template <>
struct FactorTypes<0> {
    using T = cplx;
};
template <>
struct FactorTypes<1> {
    using T = double;
};

__device__ inline cplx frcp(cplx b) {
    const double d = fma(b.re, b.re, b.im * b.im);
    return {b.re / d, -b.im / d};
}
__device__ inline double frcp(double b) { return 1.0 / b; }
__device__ inline cplx fmulx(cplx a, cplx b) {
    return {fma(-a.im, b.im, a.re * b.re), fma(a.im, b.re, a.re * b.im)};
}
__device__ inline double fmulx(double a, double b) { return a * b; }
// a - t x
__device__ inline cplx fsubx(cplx a, cplx t, cplx x) { return tmsub(a, t, x); }
__device__ inline double fsubx(double a, double t, double x) { return fma(-t, x, a); }

// a table's scalar e: its eigenvalue times its time point's ifdt, from the
// device or (ifdt null, at most two time points) by value
struct FactorScal {
    const double *eig, *ifdt;
    int64_t eig_tstride;
    double v[2];
    __device__ double at(int t, int ch) const {
        return eig[(int64_t)t * eig_tstride + ch] * (ifdt ? ifdt[t] : t ? v[1] : v[0]);
    }
};

template <int SYM, int P>
__global__ __launch_bounds__(kLane, P == 7 ? 2 : 1) void k_factor(const cplx* __restrict__ fx, FactorScal sc0, Geom geo,
                                                  int above, cplx* __restrict__ tab, int64_t tstride) {
    using T = typename FactorTypes<SYM>::T;
    constexpr int NE = P + 1;
    // slots: a divisor of kPM, so that the rounds of rows end with the partition
    constexpr int RS = P == 7 ? 8 : 12;
    static_assert(RS > P && kPM % RS == 0 && restart_round(P) % RS == 0, "slot count");
    const int g = blockIdx.x * kLane + threadIdx.x;
    const int ch = blockIdx.y, t = blockIdx.z;
    if (g >= geo.P) return;
    const int FP = factor_cols(geo);
    const double e = sc0.at(t, ch);
    // SYM 0 writes complex symmetric rows [E_1..E_P, 1/pivot] (for a symmetric
    // matrix the unit upper factor's rows are the columns of L in A = L D L^T);
    // SYM 1 writes real LU rows (forward: the multipliers of the rows below, backward: u)
    constexpr int ROW = TabFmt<T, P>::row;
    cplx* Tg = tab + ((int64_t)t * tstride + ch) * TabFmt<T, P>::units(geo) + part_col<T, P>(g);
    const int r0 = g * kPM;
    // (whole rounds of RS rows; r0 is a multiple of RS too)
    const int start = r0 > above ? r0 - above : 0;
    // column entries of the band from column `start` on
    int sc = start % kPM, gc = start / kPM;
    auto column = [&](cplx (&q)[NE]) {
        const cplx* b = fx + ((int64_t)sc * NE * FP + gc);
#pragma unroll
        for (int j = 0; j < NE; ++j) q[j] = b[j * FP];
        if (++sc == kPM) {
            sc = 0;
            ++gc;
        }
    };
    T wu[RS][NE];                    // wu[slot(r)][j] = A(r, r+j)
    double wl[SYM ? RS : 1][NE];     // wl[slot(r)][j] = A(r+j, r), j >= 1 (SYM 1)
#pragma unroll
    for (int s = 0; s < RS; ++s)
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            wu[s][j] = tzero(T{});
            if constexpr (SYM) wl[s][j] = 0.0;
        }
    auto put = [&](int slot, int j, cplx q) {
        if constexpr (SYM == 0) {
            wu[slot][j] = cplx{q.re, e * q.im};  // s + ifet r, ifet = i e
        } else {
            wu[slot][j] = fma(e, q.im, q.re);
            if (j) wl[slot][j] = fma(-e, q.im, q.re);  // antisymmetric below the diagonal
        }
    };
    cplx nx[NE];
#pragma unroll
    for (int c = 0; c < P; ++c) {  // columns start .. start+P-1 of the rows that exist
        column(nx);
#pragma unroll
        for (int j = 0; j <= c; ++j) put(c - j, j, nx[j]);
    }
    column(nx);
    // RS rows from row i on; STORE writes their table rows.  No branch inside:
    // the compiler moves updates across one to their last use, which keeps
    // every row's operands live
    auto round = [&](int i, auto store) {
#pragma unroll
        for (int s = 0; s < RS; ++s) {
            // a row at a time: later rows' column loads ahead of these products
            // would need registers for all of them
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NE; ++j) put((s + P - j) % RS, j, nx[j]);
            column(nx);
            const T rp = frcp(wu[s][0]);
            T u[NE];
#pragma unroll
            for (int k = 1; k < NE; ++k) u[k] = fmulx(wu[s][k], rp);
            if constexpr (decltype(store)::value) {
                cplx* o = Tg + (int64_t)(i + s - r0) * ROW * kLane;
                if constexpr (SYM == 0) {
#pragma unroll
                    for (int k = 1; k < NE; ++k) o[(int64_t)(k - 1) * kLane] = u[k];
                    o[(int64_t)P * kLane] = rp;
                } else {
                    put_real<P>(o, &wl[s][1], rp);
                    put_real<P>(o + TabFmt<T, P>::boff * kLane, &u[1], 1.0);
                }
            }
            // A(i+a, i+b) -= A(i+a, i) u(i, i+b)
#pragma unroll
            for (int a = 1; a < NE; ++a)
#pragma unroll
                for (int b = SYM ? 1 : a; b < NE; ++b) {
                    if constexpr (SYM == 0) {
                        T& w = wu[(s + a) % RS][b - a];
                        w = fsubx(w, wu[s][a], u[b]);
                    } else {
                        T& w = b >= a ? wu[(s + a) % RS][b - a] : wl[(s + b) % RS][a - b];
                        w = fsubx(w, wl[s][a], u[b]);
                    }
                }
        }
    };
    int i = start;
#pragma unroll 1
    for (; i < r0; i += RS) round(i, std::false_type{});
#pragma unroll 1
    for (; i < r0 + kPM; i += RS) round(i, std::true_type{});
}

// The same elimination for few tables: 16 lanes per partition, four
// partitions per wave.  A launch of one time point is bound by the chain of
// rows, and k_factor's lane issues 190 (S + e X: 130) instructions per row for
// its own partition however few waves there are.  Here lane c mod 8 of a
// partition's 16 holds column c of the window (rows i+1 .. i+8, row r in
// register r mod 8) and the pivot and the row's entries reach the others by DPP
// row broadcasts, so a row takes P products per lane instead of P(P+1)/2.  Of a
// complex symmetric matrix the lower eight lanes hold the real parts and the
// upper eight the imaginary ones (each divides one part of 1 / pivot); of a
// real one both halves hold the same.  The bits are k_factor's.  Once column i is the pivot its lane
// takes column i + 8.  The columns come from LDS, where the wave stages the
// `above` rows over its first partition and the four partitions; columns
// before the matrix are the identity's, which changes nothing below them.
// Per partition it takes four times k_factor's lane-instructions.  Measured
// against k_factor, S + i e X (S + e X), one time point: 3 tables of N = 240
// 18 us against 49 (13 against 32), 16 tables of N = 1000 19 against 41; two
// of 37 tables of N = 361 20 against 52 (81: 18 against 34).
template <int L>
__device__ inline double bcast16(double v) {  // lane L of each 16
    return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + L, 0xf, 0xf, true));
}
template <int BANKS>
__device__ inline double swap8(double v) {  // lane l ^ 8 in the banks of four lanes of BANKS, v in the others
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int l = (int)(unsigned)b, h = (int)(unsigned)(b >> 32);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(l, l, 0x128, 0xf, BANKS, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(h, h, 0x128, 0xf, BANKS, false);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
constexpr int kFactorQ = 4;  // partitions per wave
// Used up to this many waves (six per compute unit, the most its LDS holds:
// 650 waves take 18 us, 3200 78 us and 5600 118 us where k_factor takes 35 to
// 55), and this many restart rows (LDS: 50 KB)
constexpr int64_t kFactorRowWaves = 1536;
constexpr int kFactorRowAbove = 192;
// doubles per staged column, blocks of kPM columns staged for `above` restart rows
template <int P>
constexpr int factor_pe() { return P == 7 ? 8 : 10; }
inline __host__ __device__ int factor_row_blocks(int above) { return (above + kPM - 1) / kPM + kFactorQ + 1; }

// rows of partitions [g0, g0 + kFactorQ) of one table
template <int SYM, int P>
__device__ inline void factor_row(const cplx* __restrict__ fx, double e, Geom geo, int g0, int above,
                                  cplx* __restrict__ tab) {
    using T = typename FactorTypes<SYM>::T;
    constexpr int NE = P + 1, PE = factor_pe<P>();
    constexpr int ROW = TabFmt<T, P>::row;
    extern __shared__ __align__(16) double sh[];  // [2][columns][PE]: re, im or upper, lower
    const int FP = factor_cols(geo);
    const int ln = threadIdx.x, cl = ln & 7, hf = (ln >> 3) & 1;
    // stage whole blocks of kPM columns from block b0 on, a lane per (block, entry)
    const int nb = factor_row_blocks(above), b0 = g0 - (nb - kFactorQ - 1), half = nb * kPM * PE;
    for (int gb = cl; gb < nb; gb += 8)
        for (int j = ln >> 3; j < NE; j += 8) {
            const int b = b0 + gb;
            const cplx* q = fx + ((int64_t)j * FP + min(max(b, 0), FP - 1));
            cplx v[kPM];
#pragma unroll
            for (int k = 0; k < kPM; ++k) v[k] = q[(int64_t)k * NE * FP];
            double* d = sh + gb * kPM * PE + j;
#pragma unroll
            for (int k = 0; k < kPM; ++k, d += PE) {
                if (b < 0) v[k] = cplx{j == 0 ? 1.0 : 0.0, 0.0};
                if constexpr (SYM == 0) {
                    d[0] = v[k].re;
                    d[half] = e * v[k].im;
                } else {
                    const double up = fma(e, v[k].im, v[k].re);
                    d[0] = up;
                    d[half] = j ? fma(-e, v[k].im, v[k].re) : up;  // antisymmetric below the diagonal
                }
            }
        }
    __syncthreads();
    // (partitions past the last repeat it)
    const int g = min(g0 + (ln >> 4), geo.P - 1);
    const int first = (g - b0) * kPM - above;  // first row of the restarted elimination
    const double* up = sh + first * PE + (SYM == 0 ? hf * half : 0);
    const double* lo = sh + first * PE + half;
    char* Tg = (char*)(tab + part_col<T, P>(g));
    double w[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        if constexpr (SYM == 0) w[r] = r <= cl ? up[cl * PE + max(cl - r, 0)] : 0.0;
        else w[r] = r <= cl ? up[cl * PE + max(cl - r, 0)] : lo[r * PE + max(r - cl, 0)];
    }
    // eight rows from row i (of the staged columns) on, pivot columns at up / lo
    auto round = [&](int i, auto store) {
        constexpr bool STORE = decltype(store)::value;
        each(std::make_integer_sequence<int, 8>{}, [&](auto sc) {
            constexpr int S = decltype(sc)::value;
            const bool mine = cl == S;          // the pivot column's lane
            const int b1 = (cl - S - 1) & 7;    // column i + 1 + b1 (P = 7: 7 is the pivot's lane)
            const double* nu = up + (S + 8) * PE;  // column i + 8
            double a0 = w[S];
            char* o = Tg + (int64_t)(i + S - above) * ROW * kLane * 16;
            if constexpr (SYM == 0) {
                const double pr = bcast16<S>(a0), pi = bcast16<S + 8>(a0);
                if (mine) {
                    a0 = P == 8 ? nu[P] : 0.0;
#pragma unroll
                    for (int k = 0; k < 8; ++k) w[(S + 1 + k) & 7] = nu[7 - k];
                }
                // 1 / pivot = (pr - i pi) / |pivot|^2, a part in either half
                const double q0 = (hf ? -pi : pr) / fma(pr, pr, pi * pi);
                const double qr = bcast16<0>(q0), qi = bcast16<8>(q0);
                const double ar = swap8<0xc>(a0), ai = swap8<0x3>(a0);
                // u = a / pivot (k_factor's order of operations: the same bits);
                // the lower half multiplies by (re u, -im u), the upper by (im u, re u)
                const double ur = fma(-ai, qi, ar * qr), ui = fma(ai, qr, ar * qi);
                const double x1 = hf ? ui : ur, x2 = hf ? ur : -ui;
                if constexpr (STORE) {
                    *(double*)(o + (b1 * kLane * 16 + hf * 8)) = P == 7 && mine ? q0 : x1;
                    if (P == 8 && cl == 0) *(double*)(o + (P * kLane * 16 + hf * 8)) = q0;
                }
                each(std::make_integer_sequence<int, P>{}, [&](auto ac) {
                    constexpr int a = decltype(ac)::value + 1, c = (S + a) & 7;
                    double& v = w[(S + a) & 7];
                    v = fma(-bcast16<c>(a0), x1, v);
                    v = fma(-bcast16<c + 8>(a0), x2, v);
                });
            } else {
                const double* nl = lo + (S + 8) * PE;
                double l[NE];
                l[0] = bcast16<S>(a0);
#pragma unroll
                for (int a = 1; a < 8; ++a) l[a] = bcast16<S>(w[(S + a) & 7]);
                if constexpr (P == 8) l[8] = nl[8];
                // row i + 8 of the columns i + 1 .. i + 8, then column i + 8
                w[S] = nl[(7 - b1) & 7];
                if (mine) {
                    a0 = P == 8 ? nu[P] : 0.0;
#pragma unroll
                    for (int k = 0; k < 7; ++k) w[(S + 1 + k) & 7] = nu[7 - k];
                }
                const double rp = 1.0 / l[0];
                const double u = a0 * rp;
                if constexpr (STORE) {
                    if (cl == 0) put_real<P>((cplx*)o, l + 1, rp);
                    char* ob = o + (int64_t)TabFmt<T, P>::boff * kLane * 16;
                    *(double*)(ob + ((b1 >> 1) * kLane * 16 + (b1 & 1) * 8)) = P == 7 && mine ? 1.0 : u;
                    if (P == 8 && cl == 0) *(cplx*)(ob + (P / 2) * kLane * 16) = cplx{1.0, 0.0};
                }
#pragma unroll
                for (int a = 1; a < NE; ++a) w[(S + a) & 7] = fma(-l[a], u, w[(S + a) & 7]);
            }
        });
        up += 8 * PE;
        lo += 8 * PE;
    };
    int i = 0;
#pragma unroll 1
    for (; i < above; i += 8) round(i, std::false_type{});
#pragma unroll 1
    for (; i < above + kPM; i += 8) round(i, std::true_type{});
}

template <int SYM, int P>
__global__ __launch_bounds__(kLane) void k_factor_row(const cplx* __restrict__ fx, FactorScal sc, Geom geo, int above,
                                                      cplx* __restrict__ tab, int64_t tstride) {
    using T = typename FactorTypes<SYM>::T;
    const int ch = blockIdx.y, t = blockIdx.z;
    factor_row<SYM, P>(fx, sc.at(t, ch), geo, blockIdx.x * kFactorQ, above,
                       tab + ((int64_t)t * tstride + ch) * TabFmt<T, P>::units(geo));
}
// The tables, and their transfer sets, of several operators in one launch each:
// a step called by itself waits for all of them (four operators of N = 361,
// M = 9, L = 9 in turn: 115 us of its 515).
struct FactorJobs {
    FactorJob j[kFactorJobs];
    int n;
};
template <int P>
__global__ __launch_bounds__(kLane) void k_factor_jobs(FactorJobs a, Geom geo) {
    int ch = blockIdx.y, k = 0;
    while (k + 1 < a.n && ch >= a.j[k].nch) ch -= a.j[k++].nch;
    const FactorJob& J = a.j[k];
    const int t = blockIdx.z, g0 = blockIdx.x * kFactorQ;
    const double e = J.eig[ch] * (t ? J.ifdt[1] : J.ifdt[0]);
    const int64_t q = (int64_t)t * J.tstride + ch;
    if (J.real) factor_row<1, P>(J.fx, e, geo, g0, J.restart, (cplx*)J.tab + q * TabFmt<double, P>::units(geo));
    else factor_row<0, P>(J.fx, e, geo, g0, J.restart, (cplx*)J.tab + q * TabFmt<cplx, P>::units(geo));
}
template <int P>
__global__ __launch_bounds__(kLane) void k_transfer_jobs(FactorJobs a, Geom geo) {
    static_assert(trf_groups<cplx, P>() == trf_groups<double, P>(), "one grid");
    int ch = blockIdx.x, k = 0;
    while (k + 1 < a.n && ch >= a.j[k].nch) ch -= a.j[k++].nch;
    const FactorJob& J = a.j[k];
    const int64_t q = (int64_t)blockIdx.z * J.tstride + ch;
    if (J.real) transfer_cols<double, P>((const cplx*)J.tab, (double*)J.trf, geo, q);
    else transfer_cols<cplx, P>((const cplx*)J.tab, (cplx*)J.trf, geo, q);
}

// fx[(s * (p+1) + j) * FP + g] = {S, X}(c-j, c) of column c = 24 g + s, zero
// above the first row; columns from N on are the identity's (the table rows
// of the last partition's padding)
__global__ __launch_bounds__(256) void k_factor_bands(const double* __restrict__ S, const double* __restrict__ X,
                                                      cplx* __restrict__ fx, int N, int ne, int FP) {
    const int id = blockIdx.x * 256 + threadIdx.x;
    if (id >= kPM * ne * FP) return;
    const int g = id % FP, j = id / FP % ne, s = id / FP / ne;
    const int c = g * kPM + s, r = c - j;
    cplx v = {0.0, 0.0};
    if (c >= N) v.re = j == 0 ? 1.0 : 0.0;
    else if (r >= 0) v = {S[(int64_t)r * ne + j], X[(int64_t)r * ne + j]};
    fx[id] = v;
}

}  // namespace

// ---------------------------------------------------------------------------
template <int P>
static void rhs_launch(hipStream_t s, int rhs, const RhsArgs& ra, TabMap tm, const cplx* zin, cplx* vout, int nch,
                       Geom geo) {
    dim3 rgrid((geo.N + 255) / 256, nch);
    dim3 sgrid((geo.N + 255) / 256, (nch + kRhsCG - 1) / kRhsCG);
    switch (rhs) {
        case RHS_CBAND: hipLaunchKernelGGL(k_rhs<P>, rgrid, dim3(256), 0, s, ra, tm, zin, vout, geo.N); break;
        case RHS_RBAND:
            hipLaunchKernelGGL((k_rhs_shared<RHS_RBAND, P>), sgrid, dim3(256), 0, s, ra, zin, vout, geo.N, nch);
            break;
        case RHS_SX_SYM:
            hipLaunchKernelGGL((k_rhs_shared<RHS_SX_SYM, P>), sgrid, dim3(256), 0, s, ra, zin, vout, geo.N, nch);
            break;
        case RHS_SX_ASY:
            hipLaunchKernelGGL((k_rhs_shared<RHS_SX_ASY, P>), sgrid, dim3(256), 0, s, ra, zin, vout, geo.N, nch);
            break;
        default: break;
    }
}

void launch_rhs(hipStream_t s, int rhs, const RhsArgs& ra, TabMap tm, const cplx* zin, cplx* vout, int nch, Geom geo) {
    if (geo.hw == 8) rhs_launch<8>(s, rhs, ra, tm, zin, vout, nch, geo);
    else rhs_launch<7>(s, rhs, ra, tm, zin, vout, nch, geo);
}

// Largest grid whose solves run staged (geo.stage_grid, default kStageGrid):
// eight waves per work-group, part of the table in LDS and the right-hand side
// formed in the launch.  One such work-group fills a CU (133-156 KB of LDS), so
// up to 256 run at once and up to 512 in two rounds; larger grids run one wave
// per work-group, four per CU.  Batched shots, 16 steps, N = 1200, staged
// against one wave: 240 channels 4.61 / 5.75 ms, 320 channels 6.80 / 6.49,
// 480 channels 7.92 / 7.96, 640 channels 11.2 / 10.0.

// Partitions per segment: one segment when the channel fits a work-group (no
// halo to run), else the fewest segments that hold them with their halos,
// plus geo.seg_add, none empty
static int seg_parts(const Geom& geo, int pk) {
    const int smax = seg_max(pk), fewest = (geo.P + smax - 1) / smax;
    int nseg = (geo.P <= kLane ? 1 : fewest) + std::max(0, geo.seg_add);
    if (nseg > 1) nseg = std::max(nseg, fewest);
    nseg = std::min(geo.P, nseg);
    return (geo.P + nseg - 1) / nseg;
}

void solve_order(const int* tab, int nch, int nseg, int* order) {
    // (table, segment, channel) ascending, dealt to the XCDs in contiguous
    // chunks; XCD x's k-th work-group has linear id x + kXcds k
    std::vector<int> e((size_t)nch * nseg);
    for (int ch = 0; ch < nch; ++ch)
        for (int sg = 0; sg < nseg; ++sg) e[(size_t)ch * nseg + sg] = ch * nseg + sg;
    std::stable_sort(e.begin(), e.end(), [&](int a, int b) {
        const int ta = tab[a / nseg], tb = tab[b / nseg];
        if (ta != tb) return ta < tb;
        return a % nseg < b % nseg;
    });
    const int T = nch * nseg, base = T / kXcds, extra = T % kXcds;
    int j = 0;
    for (int x = 0; x < kXcds; ++x) {
        const int n = base + (x < extra ? 1 : 0);
        for (int k = 0; k < n; ++k) {
            const int q = e[j++];
            order[x + kXcds * k] = (q / nseg) << 8 | q % nseg;
        }
    }
}

// The launch of the solve with eight lanes per partition: channels of at most
// kSplitParts partitions always run it, longer ones if they can be cut into
// work-groups of that many partitions, halos included, of which no more than
// kSplitGrid result (the outer segments have a halo on one side only and own
// that many more partitions).  One step, N = 1000, k_bsolve against eight lanes:
// 100 channels (200 work-groups) 184 / 152 us, 128 (256) 194 / 166, 140 (280)
// 200 / 214; N = 1500: 80 channels (240) 183 / 149, 86 (258) 186 / 195 (with the
// work-groups of one table on one XCD the cut ones take 150, 160 and 146).
//
// Within these work-groups, the fewest segments that leave each the fewest
// waves (short channels too, unless the solve is in place, where one segment
// keeps the right-hand side in the launch): a step of 8 channels of N = 1000
// takes 105 us with four waves each, 99 / 94 / 87 as the operators' solves come
// down to three and two, and does not change in between.
struct SplitGrid {
    int nseg = 0, sn = 0, sx = 0, parts = 0;  // nseg 0: not this launch; parts: the most of a work-group
    int waves() const { return (parts + 7) / 8; }
};
static SplitGrid split_grid(const Geom& geo, int nch, int pk, bool in_place) {
    const bool whole = geo.P <= kSplitParts;
    auto cut = [&](int n) {
        SplitGrid g;
        const int w = (geo.P + 2 * pk * (n - 1) + n - 1) / n, sn = w - 2 * pk;
        if (w <= kSplitParts && sn >= 1 && pk + (n - 1) * sn < geo.P) g = {n, sn, pk, w};
        return g;
    };
    SplitGrid best;
    if (!whole || !in_place) {
        const int most = (int)std::min<int64_t>(geo.P, std::min(kSplitGrid, geo.stage_grid) / std::max(1, nch));
        int waves = whole ? (geo.P + 7) / 8 : kSplitParts / 8 + 1;
        for (int n = 2; n <= most; ++n) {
            const SplitGrid g = cut(n);
            if (g.nseg && g.waves() < waves) {
                best = g;
                waves = g.waves();
            }
        }
        if (best.nseg && geo.seg_add > 0 && best.nseg + geo.seg_add <= most) {
            const SplitGrid g = cut(best.nseg + geo.seg_add);
            if (g.nseg) best = g;
        }
    }
    if (whole && !best.nseg) {
        best.sn = seg_parts(geo, pk);
        best.nseg = (geo.P + best.sn - 1) / best.sn;
        best.parts = std::min(geo.P, best.nseg > 1 ? best.sn + 2 * pk : best.sn);
    }
    return best;
}

// (The count is the launch's own, cut or not, so that an order built for it is
// used: a cut launch is bound by its loads, and without the order the channels
// of one table lie on different XCDs.  31 channels of N = 1000, HBM reads per R /
// D / free launch 6.1 / 6.5 / 17.3 -> 2.6 / 3.7 / 5.5 MB, a step of a run 106.8 ->
// 105.1 us; 41 of N = 1500 120.5 -> 117.4, 128 of N = 1000 165.7 -> 160.5.)
int solve_segments(const Geom& geo, int nch, int pk, bool in_place) {
    if (pk > kPKMax) return 0;  // the sequential solve: no segments
    const SplitGrid g8 = split_grid(geo, nch, pk, in_place);
    if (g8.nseg) return g8.nseg;
    const int sn = seg_parts(geo, pk);
    return (geo.P + sn - 1) / sn;
}

template <class TF, int ROLE, int P>
static void bsolve(hipStream_t s, const TF* tab, const TF* trf, TabMap tm, const cplx* zin, cplx* vbuf,
                   cplx* zout, int nch, Geom geo, const RhsArgs& ra, int pk) {
    const int PK = pk > 0 ? pk : (ROLE == RHS_SX_ASY ? kPKD : kPKS);
    if (PK > kPKMax) {
        // the carry would reach further than a work-group holds: sequential solve
        rhs_launch<P>(s, ROLE, ra, tm, zin, vbuf, nch, geo);
        hipLaunchKernelGGL((k_seqsolve<TF, P>), dim3((nch + 63) / 64), dim3(64), 0, s, (const cplx*)tab, tm, vbuf, zout,
                           geo, nch);
        return;
    }
    const SplitGrid g8 = split_grid(geo, nch, PK, zin == zout);
    const int sn = g8.nseg ? g8.sn : seg_parts(geo, PK);
    const int nseg = g8.nseg ? g8.nseg : (geo.P + sn - 1) / sn;
    if (tm.order && nseg != tm.order_nseg) tm.order = nullptr;  // built for another launch shape
    // z and x apart: another work-group never reads rows of z that one writes
    const uintptr_t a0 = (uintptr_t)zin, b0 = (uintptr_t)zout, len = sizeof(cplx) * (uintptr_t)nch * geo.N;
    const bool apart = a0 + len <= b0 || b0 + len <= a0;
    const dim3 grid(nseg, nch);
    if (g8.nseg) {
        const dim3 block((g8.parts + 7) / 8 * kLane);
        if (apart || (nseg == 1 && a0 == b0)) {
            hipLaunchKernelGGL((k_bsolve8<TF, ROLE, true, P>), grid, block, 0, s, (const cplx*)tab, trf, tm, zin, zout,
                               geo, sn, g8.sx, PK, ra);
            return;
        }
        rhs_launch<P>(s, ROLE, ra, tm, zin, vbuf, nch, geo);
        hipLaunchKernelGGL((k_bsolve8<TF, ROLE, false, P>), grid, block, 0, s, (const cplx*)tab, trf, tm, vbuf, zout,
                           geo, sn, g8.sx, PK, RhsArgs{});
        return;
    }
    const bool staged = (int64_t)nseg * nch <= geo.stage_grid;
    if (staged && apart) {
        hipLaunchKernelGGL((k_bsolve<TF, ROLE, true, true, P>), grid, dim3(kLane * kWavesStaged), 0, s,
                           (const cplx*)tab, trf, tm, zin, zout, geo, sn, PK, ra);
        return;
    }
    rhs_launch<P>(s, ROLE, ra, tm, zin, vbuf, nch, geo);
    if (staged)
        hipLaunchKernelGGL((k_bsolve<TF, ROLE, true, false, P>), grid, dim3(kLane * kWavesStaged), 0, s,
                           (const cplx*)tab, trf, tm, vbuf, zout, geo, sn, PK, RhsArgs{});
    else
        hipLaunchKernelGGL((k_bsolve<TF, ROLE, false, false, P>), grid, dim3(kLane), 0, s, (const cplx*)tab, trf, tm,
                           vbuf, zout, geo, sn, PK, RhsArgs{});
}

template <class TF, int ROLE>
static void bsolve_w(hipStream_t s, const TF* tab, const TF* trf, TabMap tm, const cplx* zin, cplx* vbuf, cplx* zout,
                     int nch, Geom geo, const RhsArgs& ra, int pk) {
    if (geo.hw == 8) bsolve<TF, ROLE, 8>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
    else bsolve<TF, ROLE, 7>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
}

void launch_rsolve_c(hipStream_t s, int role, const RhsArgs& ra, const cplx* tab, const cplx* trf, TabMap tm,
                     const cplx* zin, cplx* vbuf, cplx* zout, int nch, Geom geo, int pk) {
    if (role == RHS_CBAND) bsolve_w<cplx, RHS_CBAND>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
    else bsolve_w<cplx, RHS_SX_SYM>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
}
void launch_rsolve_r(hipStream_t s, int role, const RhsArgs& ra, const double* tab, const double* trf, TabMap tm,
                     const cplx* zin, cplx* vbuf, cplx* zout, int nch, Geom geo, int pk) {
    if (role == RHS_RBAND) bsolve_w<double, RHS_RBAND>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
    else bsolve_w<double, RHS_SX_ASY>(s, tab, trf, tm, zin, vbuf, zout, nch, geo, ra, pk);
}

void launch_transfer_c(hipStream_t s, const cplx* tab, cplx* trf, int ntab, Geom geo) {
    launch_transfer_c(s, tab, trf, ntab, 1, 0, geo);
}
template <class TF, int P>
static void transfer_launch(hipStream_t s, const void* tab, TF* trf, int per_t, int nt, int64_t stride, Geom geo) {
    hipLaunchKernelGGL((k_transfer<TF, P>), dim3(per_t, geo.NG * trf_groups<TF, P>(), nt), dim3(kLane), 0, s,
                       (const cplx*)tab, trf, geo, stride);
}
void launch_transfer_c(hipStream_t s, const cplx* tab, cplx* trf, int per_t, int nt, int64_t stride, Geom geo) {
    if (geo.hw == 8) transfer_launch<cplx, 8>(s, tab, trf, per_t, nt, stride, geo);
    else transfer_launch<cplx, 7>(s, tab, trf, per_t, nt, stride, geo);
}
void launch_transfer_r(hipStream_t s, const double* tab, double* trf, int ntab, Geom geo) {
    if (geo.hw == 8) transfer_launch<double, 8>(s, tab, trf, ntab, 1, 0, geo);
    else transfer_launch<double, 7>(s, tab, trf, ntab, 1, 0, geo);
}

void launch_tab_ldlt(hipStream_t s, const cplx* lower, cplx* tab, int nl, Geom geo) {
    if (geo.hw == 8) hipLaunchKernelGGL(k_tab_ldlt<8>, dim3(geo.NG, nl), dim3(kLane), 0, s, lower, tab, geo);
    else hipLaunchKernelGGL(k_tab_ldlt<7>, dim3(geo.NG, nl), dim3(kLane), 0, s, lower, tab, geo);
}
void launch_tab_chol(hipStream_t s, const double* chol, double* tab, Geom geo) {
    if (geo.hw == 8) hipLaunchKernelGGL(k_tab_chol<8>, dim3(geo.NG), dim3(kLane), 0, s, chol, (cplx*)tab, geo);
    else hipLaunchKernelGGL(k_tab_chol<7>, dim3(geo.NG), dim3(kLane), 0, s, chol, (cplx*)tab, geo);
}

void launch_band_diag_r(hipStream_t s, const double* src, double* dst, int n, int N, int p) {
    const int64_t total = (int64_t)n * (p + 1) * N;
    hipLaunchKernelGGL(k_band_diag<double>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, src, dst, total, N,
                       p + 1);
}
void launch_band_pair(hipStream_t s, const double* S, const double* X, cplx* dst, int N, int p) {
    const int64_t total = (int64_t)(p + 1) * N;
    hipLaunchKernelGGL(k_band_pair, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, S, X, dst, total);
}
void launch_band_diag_c(hipStream_t s, const cplx* src, cplx* dst, int n, int N, int p) {
    const int64_t total = (int64_t)n * (p + 1) * N;
    hipLaunchKernelGGL(k_band_diag<cplx>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, src, dst, total, N,
                       p + 1);
}

void launch_factor_bands(hipStream_t s, const double* S, const double* X, cplx* fx, Geom geo) {
    const int total = kPM * (geo.hw + 1) * factor_cols(geo);
    hipLaunchKernelGGL(k_factor_bands, dim3((total + 255) / 256), dim3(256), 0, s, S, X, fx, geo.N, geo.hw + 1,
                       factor_cols(geo));
}
// waves and restart rows within k_factor_row's range
static int row_groups(const Geom& geo) { return (geo.P + kFactorQ - 1) / kFactorQ; }
static bool row_fits(const Geom& geo, int64_t tables, int above) {
    return row_groups(geo) * tables <= kFactorRowWaves && above <= kFactorRowAbove;
}
template <int P>
static size_t row_lds(int above) { return sizeof(double) * 2 * factor_row_blocks(above) * kPM * factor_pe<P>(); }

template <int SYM, int P>
static void factor_launch_p(hipStream_t s, const cplx* fx, const FactorScal& sc, int nt, int nch, Geom geo, cplx* tab,
                            int restart, int64_t ts) {
    const int above = restart_rows(P, restart);
    if (row_fits(geo, (int64_t)nch * nt, above))
        hipLaunchKernelGGL((k_factor_row<SYM, P>), dim3(row_groups(geo), nch, nt), dim3(kLane), row_lds<P>(above), s, fx,
                           sc, geo, above, tab, ts);
    else
        hipLaunchKernelGGL((k_factor<SYM, P>), dim3(geo.NG, nch, nt), dim3(kLane), 0, s, fx, sc, geo, above,
                           tab, ts);
}
template <int SYM>
static void factor_launch(hipStream_t s, const cplx* fx, const FactorScal& sc, int nt, int nch, Geom geo, cplx* tab,
                          int restart, int64_t ts) {
    if (geo.hw == 8) factor_launch_p<SYM, 8>(s, fx, sc, nt, nch, geo, tab, restart, ts);
    else factor_launch_p<SYM, 7>(s, fx, sc, nt, nch, geo, tab, restart, ts);
}
void launch_factor_sym(hipStream_t s, const cplx* fx, const double* eig, const double* ifdt, int nt, int nch, Geom geo,
                       cplx* tab, int64_t eig_tstride, int restart, int64_t tab_tstride) {
    factor_launch<0>(s, fx, FactorScal{eig, ifdt, eig_tstride, {}}, nt, nch, geo, tab, restart,
                     tab_tstride > 0 ? tab_tstride : nch);
}
void launch_factor_asy(hipStream_t s, const cplx* fx, const double* eig, const double* ifdt, int nt, int nch, Geom geo,
                       double* tab, int64_t eig_tstride, int restart) {
    factor_launch<1>(s, fx, FactorScal{eig, ifdt, eig_tstride, {}}, nt, nch, geo, (cplx*)tab, restart, nch);
}

template <int P>
static void factor_jobs(hipStream_t s, const FactorJobs& a, int nt, const Geom& geo) {
    int rows = 0, above = 0;
    bool fit = true;  // each by itself: together they take no longer than one after the other
    for (int k = 0; k < a.n; ++k) {
        rows += a.j[k].nch;
        above = std::max(above, a.j[k].restart);
        fit = fit && row_fits(geo, (int64_t)a.j[k].nch * nt, a.j[k].restart);
    }
    if (fit) {
        hipLaunchKernelGGL(k_factor_jobs<P>, dim3(row_groups(geo), rows, nt), dim3(kLane), row_lds<P>(above), s, a, geo);
        hipLaunchKernelGGL(k_transfer_jobs<P>, dim3(rows, geo.NG * trf_groups<cplx, P>(), nt), dim3(kLane), 0, s, a, geo);
        return;
    }
    for (int k = 0; k < a.n; ++k) {
        const FactorJob& J = a.j[k];
        const FactorScal sc{J.eig, nullptr, 0, {J.ifdt[0], J.ifdt[1]}};
        const dim3 tg(J.nch, geo.NG * trf_groups<cplx, P>(), nt);
        if (J.real) {
            factor_launch_p<1, P>(s, J.fx, sc, nt, J.nch, geo, (cplx*)J.tab, J.restart, J.tstride);
            hipLaunchKernelGGL((k_transfer<double, P>), tg, dim3(kLane), 0, s, (const cplx*)J.tab, (double*)J.trf, geo,
                               J.tstride);
        } else {
            factor_launch_p<0, P>(s, J.fx, sc, nt, J.nch, geo, (cplx*)J.tab, J.restart, J.tstride);
            hipLaunchKernelGGL((k_transfer<cplx, P>), tg, dim3(kLane), 0, s, (const cplx*)J.tab, (cplx*)J.trf, geo,
                               J.tstride);
        }
    }
}
void launch_factor_jobs(hipStream_t s, const FactorJob* jobs, int n, int nt, Geom geo) {
    FactorJobs a{};
    for (int k = 0; k < n && a.n < kFactorJobs; ++k)
        if (jobs[k].nch > 0) {
            a.j[a.n] = jobs[k];
            a.j[a.n].restart = restart_rows(geo.hw, jobs[k].restart);
            ++a.n;
        }
    if (a.n == 0) return;
    if (geo.hw == 8) factor_jobs<8>(s, a, nt, geo);
    else factor_jobs<7>(s, a, nt, geo);
}

// ---------------------------------------------------------------------------
// host: reach of the recurrences (qpc_solve.h)
namespace {
struct hc {
    double re, im;
};
inline hc hmul(hc a, hc b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
inline hc hsub(hc a, hc b) { return {a.re - b.re, a.im - b.im}; }
inline hc hdiv(hc a, hc b) {
    const double d = b.re * b.re + b.im * b.im;
    return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}
inline double habs(hc a) { return std::sqrt(a.re * a.re + a.im * a.im); }

// rows from a unit source until the response of L^-1 (fwd) or U^-1 (bwd)
// stays below tol times its peak, in the window [w0, w0 + W) of A
Reach window_reach(const double* S, const double* X, int p, double e, int asym, int w0, int W, double tol) {
    const int ne = p + 1;
    // A(i, j) in the window, banded: U rows (unit diagonal after scaling) and L multipliers
    auto upper = [&](int i, int k) -> hc {  // A(i, i+k), k >= 0
        const double sv = S[(size_t)(w0 + i) * ne + k], xv = X[(size_t)(w0 + i) * ne + k];
        return asym ? hc{sv + e * xv, 0.0} : hc{sv, e * xv};
    };
    auto lower = [&](int i, int k) -> hc {  // A(i+k, i), k >= 1
        const double sv = S[(size_t)(w0 + i) * ne + k], xv = X[(size_t)(w0 + i) * ne + k];
        return asym ? hc{sv - e * xv, 0.0} : hc{sv, e * xv};
    };
    // dense-banded LU without pivoting: U[i][k] = U(i, i+k), Lm[i][k] = L(i+k, i)
    std::vector<hc> U((size_t)W * ne), Lm((size_t)W * ne);
    std::vector<hc> row(2 * p + 1);
    for (int i = 0; i < W; ++i) {
        // row i of A from column i-p to i+p, minus the eliminated rows above
        for (int c = -p; c <= p; ++c) {
            const int j = i + c;
            hc v = {0.0, 0.0};
            if (j >= 0 && j < W) v = c >= 0 ? (c <= p ? upper(i, c) : hc{0, 0}) : lower(j, -c);
            row[c + p] = v;
        }
        for (int k = std::max(0, i - p); k < i; ++k) {
            // eliminate column k with U row k: l = row[k] / U(k,k)
            const hc l = hdiv(row[k - i + p], U[(size_t)k * ne]);
            Lm[(size_t)k * ne + (i - k)] = l;
            for (int c = 0; c <= p && k + c < W; ++c) {
                const int col = k + c - i + p;
                if (col > k - i + p && col <= 2 * p) row[col] = hsub(row[col], hmul(l, U[(size_t)k * ne + c]));
            }
            row[k - i + p] = {0.0, 0.0};
        }
        for (int c = 0; c <= p; ++c) U[(size_t)i * ne + c] = (i + c < W) ? row[c + p] : hc{0.0, 0.0};
    }
    const int src = std::min(60, W / 4);
    Reach r{0, 0, 0};
    // restarted elimination: the same LU begun afresh at row src (rows above
    // it dropped, as k_factor restarts above each partition); rst is the
    // distance after which its U rows stay within 1e-14 of the row's largest
    // entry from the full elimination's (the difference falls about three
    // decades per 24 rows to a few ulps, where rounding keeps it until the
    // two eliminations become bit-identical some 110-130 rows on)
    {
        std::vector<hc> Ur((size_t)W * ne);
        int last = src;
        for (int i = src; i < W; ++i) {
            for (int c = -p; c <= p; ++c) {
                const int j = i + c;
                hc v = {0.0, 0.0};
                if (j >= src && j < W) v = c >= 0 ? upper(i, c) : lower(j, -c);
                row[c + p] = v;
            }
            for (int k = std::max(src, i - p); k < i; ++k) {
                const hc l = hdiv(row[k - i + p], Ur[(size_t)k * ne]);
                for (int c = 0; c <= p && k + c < W; ++c) {
                    const int col = k + c - i + p;
                    if (col > k - i + p && col <= 2 * p) row[col] = hsub(row[col], hmul(l, Ur[(size_t)k * ne + c]));
                }
                row[k - i + p] = {0.0, 0.0};
            }
            double big = 0.0, dif = 0.0;
            for (int c = 0; c <= p; ++c) {
                Ur[(size_t)i * ne + c] = (i + c < W) ? row[c + p] : hc{0.0, 0.0};
                big = std::max(big, habs(U[(size_t)i * ne + c]));
                dif = std::max(dif, habs(hsub(Ur[(size_t)i * ne + c], U[(size_t)i * ne + c])));
            }
            if (dif > 1e-14 * big) last = i;
        }
        r.rst = last - src + 1;
    }
    // forward: L y = e_src (unit lower)
    {
        std::vector<hc> y(W, hc{0.0, 0.0});
        y[src] = {1.0, 0.0};
        double peak = 1.0;
        int last = src;
        std::vector<double> mag(W, 0.0);
        for (int i = src + 1; i < W; ++i) {
            hc v = {0.0, 0.0};
            for (int k = 1; k <= p && i - k >= src; ++k) v = hsub(v, hmul(Lm[(size_t)(i - k) * ne + k], y[i - k]));
            y[i] = v;
            mag[i] = habs(v);
            peak = std::max(peak, mag[i]);
        }
        for (int i = src + 1; i < W; ++i)
            if (mag[i] > tol * peak) last = i;
        r.fwd = last - src;
    }
    // backward: (D^-1 U) x = e_src (unit upper)
    {
        const int sb = W - 1 - src;
        std::vector<hc> x(W, hc{0.0, 0.0});
        std::vector<double> mag(W, 0.0);
        x[sb] = {1.0, 0.0};
        double peak = 1.0;
        int first = sb;
        for (int i = sb - 1; i >= 0; --i) {
            hc v = {0.0, 0.0};
            const hc d = U[(size_t)i * ne];
            for (int k = 1; k <= p && i + k <= sb; ++k) v = hsub(v, hmul(hdiv(U[(size_t)i * ne + k], d), x[i + k]));
            x[i] = v;
            mag[i] = habs(v);
            peak = std::max(peak, mag[i]);
        }
        for (int i = sb - 1; i >= 0; --i)
            if (mag[i] > tol * peak) first = i;
        r.bwd = sb - first;
    }
    return r;
}
}  // namespace

Reach solve_reach(const double* S, const double* X, int N, int p, double e, int asym, double tol) {
    const int W = std::min(N, 900);
    Reach a = window_reach(S, X, p, e, asym, 0, W, tol);
    if (N > W)
        for (int w0 : {(N - W) / 2, N - W}) {
            const Reach b = window_reach(S, X, p, e, asym, w0, W, tol);
            a.fwd = std::max(a.fwd, b.fwd);
            a.bwd = std::max(a.bwd, b.bwd);
            a.rst = std::max(a.rst, b.rst);
        }
    return a;
}

DPlan coupling_plan(const double* S, const double* X, int N, int p, double emax, int asym) {
    DPlan d{asym ? kPKD : kPKS, kRestart};
    if (!(emax > 0.0)) return d;
    int reach = 0, rst = 0;
    for (double f : {1.0, 0.5, 0.25, 0.0}) {
        const Reach r = solve_reach(S, X, N, p, emax * f, asym);
        reach = std::max(reach, std::max(r.fwd, r.bwd));
        rst = std::max(rst, r.rst);
    }
    const int W = std::min(N, 900);
    const int NP = (N + kPM - 1) / kPM;
    int pk = (reach + kPM - 1) / kPM + 1;
    if (reach + std::min(60, W / 4) + 1 >= W) {
        // the response had not decayed inside the window: a carry over every
        // partition of the channel is exact when the whole operator was the
        // window, else nothing short of the sequential solve is
        pk = W == N ? NP - 1 : kPKMax + 1;
    }
    if (pk >= NP - 1) pk = std::max(NP - 1, 1);  // the carry reaches the channel start: exact
    if (pk > kPKMax) pk = kPKMax + 1;
    d.pk = std::max(pk, std::min(kPKS, std::max(NP - 1, 1)));
    d.restart = std::max(kRestart, (rst + 15) / 16 * 16);
    return d;
}

}  // namespace qpc
