// qpc_krylov.hip -- device pieces of the Krylov propagator (gfx950).
//
// A Lanczos vector of a small grid is bound by what lies between its kernels,
// not by them: two host round trips for its products and norm, with their
// copies, took half of its 119 us (N = 600, L = 12).  The chain therefore
// stays on the device: the products of k_dots are summed where k_axpy_norm
// uses them, the norms it leaves per channel are summed by the next vector's
// k_hmul, which also normalises the vector, and the tridiagonal goes to host
// memory that the device writes.  The order of every sum is fixed and does not
// depend on the launch shape.  A vector now takes 34 us, 30 of them in its four
// kernels: k_hmul 4.9, k_dots 4.4, k_ssolve 11.4, k_axpy_norm 9.0 (N = 3000,
// L = 81: 163 -> 91 us).
#include "qpc_krylov.h"

#include <algorithm>

namespace qpc {
namespace {

constexpr int kTile = 128;         // rows per work-group of k_hmul
constexpr int kNormThreads = 1024; // rows of a channel at a time in k_axpy_norm
constexpr int kNormSums = 256;     // partial sums of a channel's norm (rows i mod 256)

// a x + t, component by component
__device__ inline cplx band_fma(double a, cplx x, cplx t) { return {fma(a, x.re, t.re), fma(a, x.im, t.im)}; }

// b_k from the squared norm (orthogonalize_ip, la_1e.hpp:195-240: below 1e-13
// the subspace ends; the first vector's is always used); the channels in order
__device__ inline double norm_of(const double* __restrict__ npart, int nch, int first) {
    double s = 0.0;
#pragma unroll 16
    for (int i = 0; i < nch; ++i) s += npart[i];
    return !first && s < 1e-13 ? 0.0 : sqrt(s);
}

// u = v / |v|, t = H(az) u over every channel: H_l u, then the couplings from
// the channels l - 1 (F, G) and l + 1 (G, F) of u, each banded product from the
// lowest diagonal's neighbour outwards (i - 1 .. i - P, then i .. i + P).  A
// row's operands are 3 (2 P + 1) band entries, all requested before their first
// use, and the three channels' rows from LDS.
template <int P>
__global__ __launch_bounds__(kTile) void k_hmul(const double* __restrict__ Hd, const double* __restrict__ Fd,
                                                const double* __restrict__ Gd, const double* __restrict__ y10,
                                                const double* __restrict__ q10, double az, int L, int m0, int N,
                                                const cplx* __restrict__ v, const double* __restrict__ npart, int nch,
                                                int first, double* b_out, cplx* __restrict__ u, cplx* __restrict__ t) {
    constexpr int NX = kTile + 2 * P;
    __shared__ cplx sx[3][NX];  // channels l - 1, l, l + 1 of u
    const int tid = threadIdx.x, r0 = blockIdx.x * kTile, i = r0 + tid;
    const int ch = blockIdx.y, il = ch % L;
    const int m = m0 + ch / L, l = il + (m < 0 ? -m : m);
    const int ic = min(i, N - 1);
    const double* H = Hd + (int64_t)l * (P + 1) * N;
    double hu[P + 1], fu[P + 1], gu[P + 1], hl[P], fl[P], gl[P];
#pragma unroll
    for (int k = 0; k <= P; ++k) {
        hu[k] = H[(int64_t)k * N + ic];
        fu[k] = Fd[(int64_t)k * N + ic];
        gu[k] = Gd[(int64_t)k * N + ic];
        if (ic + k >= N) hu[k] = fu[k] = gu[k] = 0.0;  // past the matrix, whatever the caller's arrays hold there
    }
#pragma unroll
    for (int j = 1; j <= P; ++j) {
        const int64_t o = (int64_t)j * N + max(ic - j, 0);
        hl[j - 1] = H[o];
        fl[j - 1] = Fd[o];
        gl[j - 1] = Gd[o];
    }
    const bool lo = il > 0, hi = il < L - 1;
    const double qm = lo ? az * q10[ch - 1] : 0.0, ym = lo ? az * y10[ch - 1] : 0.0;
    const double qp = hi ? az * q10[ch] : 0.0, yp = hi ? az * y10[ch] : 0.0;
    const cplx* x = v + (int64_t)ch * N;
    const cplx zero = {0.0, 0.0};
    cplx xc[2], xm[2], xp[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = r0 - P + tid + k * kTile;
        const bool in = r >= 0 && r < N && tid + k * kTile < NX;
        const int rc = in ? r : 0;
        xc[k] = x[rc];
        xm[k] = x[rc - (lo ? N : 0)];
        xp[k] = x[rc + (hi ? N : 0)];
        if (!in) xc[k] = zero;
        if (!in || !lo) xm[k] = zero;
        if (!in || !hi) xp[k] = zero;
    }
    const double nk = norm_of(npart, nch, first);
    if (blockIdx.x == 0 && ch == 0 && tid == 0) *b_out = nk;
    const double inv = nk == 0.0 ? 0.0 : 1.0 / nk;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int e = tid + k * kTile;
        if (e < NX) {
            sx[0][e] = xm[k] * inv;
            sx[1][e] = xc[k] * inv;
            sx[2][e] = xp[k] * inv;
        }
    }
    __syncthreads();
    if (i >= N) return;
    cplx h = zero, fm = zero, gm = zero, fp = zero, gp = zero;
#pragma unroll
    for (int j = 1; j <= P; ++j) {
        const int e = tid + P - j;
        h = band_fma(hl[j - 1], sx[1][e], h);
        fm = band_fma(fl[j - 1], sx[0][e], fm);
        gm = band_fma(-gl[j - 1], sx[0][e], gm);
        fp = band_fma(fl[j - 1], sx[2][e], fp);
        gp = band_fma(-gl[j - 1], sx[2][e], gp);
    }
#pragma unroll
    for (int k = 0; k <= P; ++k) {
        const int e = tid + P + k;
        h = band_fma(hu[k], sx[1][e], h);
        fm = band_fma(fu[k], sx[0][e], fm);
        gm = band_fma(gu[k], sx[0][e], gm);
        fp = band_fma(fu[k], sx[2][e], fp);
        gp = band_fma(gu[k], sx[2][e], gp);
    }
    // + i qm F u(l-1) - i ym G u(l-1) - i yp G u(l+1) - i qp F u(l+1)
    h = {fma(-qm, fm.im, h.re), fma(qm, fm.re, h.im)};
    h = {fma(ym, gm.im, h.re), fma(-ym, gm.re, h.im)};
    h = {fma(yp, gp.im, h.re), fma(-yp, gp.re, h.im)};
    h = {fma(qp, fp.im, h.re), fma(-qp, fp.re, h.im)};
    u[(int64_t)ch * N + i] = sx[1][tid + P];
    t[(int64_t)ch * N + i] = h;
}

__global__ void k_norm_final(const double* __restrict__ npart, int nch, double* b_out) {
    const double b = norm_of(npart, nch, 0);
    if (threadIdx.x == 0) *b_out = b;
}

// sum of 256 values s[0..255] by halves (i + 128, i + 64, ..): lane 0 of the
// first wave has it
__device__ inline double half_sum(const double* s) {
    const int l = threadIdx.x;
    double v = (s[l] + s[l + 128]) + (s[l + 64] + s[l + 192]);
#pragma unroll
    for (int st = 32; st > 0; st >>= 1) v += __shfl_down(v, st);
    return v;
}

// partial b of vector vi at part[b * k + vi]: block b's chunk of the rows, a
// thread the rows e0 + tid + 256 n in order, the threads by halves
__global__ __launch_bounds__(256) void k_dots(const cplx* __restrict__ U, int64_t stride, const cplx* __restrict__ v,
                                              int64_t n, cplx* __restrict__ part) {
    __shared__ double sre[256], sim[256];
    const int b = blockIdx.x, vi = blockIdx.y;
    const cplx* u = U + (int64_t)vi * stride;
    const int64_t chunk = (n + kDotBlocks - 1) / kDotBlocks;
    const int64_t e0 = (int64_t)b * chunk, e1 = e0 + chunk < n ? e0 + chunk : n;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) {
        const cplx a = u[e], c = v[e];
        re += fma(a.re, c.re, a.im * c.im);
        im += fma(a.re, c.im, -(a.im * c.re));
    }
    sre[threadIdx.x] = re;
    sim[threadIdx.x] = im;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    re = half_sum(sre);
    im = half_sum(sim);
    if (threadIdx.x == 0) part[(int64_t)b * gridDim.y + vi] = cplx{re, im};
}

// |c|^2 > 4e-27 as two products and their sum
__device__ inline bool coef_used(cplx c) {
#pragma clang fp contract(off)
    const double a = c.re * c.re, b = c.im * c.im;
    return a + b > 4e-27;
}

// v -= sum_{i<k} c_i U_i with c_i the sum of k_dots' partials in order, left
// out where |c_i|^2 <= 4e-27 (the last is always used); a_out = Re c_{k-1};
// then the channel's <v|S|v>: a row's product with S from i - 1 .. i - P, then
// i .. i + P; rows i mod 256 in order, these by halves.  One work-group per
// channel (k = 0: only the norm of v).
template <int P>
__global__ __launch_bounds__(kNormThreads) void k_axpy_norm(const cplx* __restrict__ U, int64_t stride, int k,
                                                            const double* __restrict__ part, double* a_out,
                                                            const double* __restrict__ Sd, cplx* v, int N,
                                                            double* __restrict__ npart) {
    __shared__ cplx sc[256];
    __shared__ int si[256], cnt[4];
    __shared__ double sd[kNormThreads];
    const int tid = threadIdx.x, ch = blockIdx.x;
    const int64_t o = (int64_t)ch * N;
    cplx* x = v + o;
    if (k > 0) {
        if (tid < 2 * k) {
            double s = 0.0;
#pragma unroll 32
            for (int q = 0; q < kDotBlocks; ++q) s += part[(int64_t)q * 2 * k + tid];
            sd[tid] = s;
        }
        __syncthreads();
        // the coefficients in use, compacted in order (k <= 256)
        cplx c = {0.0, 0.0};
        if (tid < k) c = {sd[2 * tid], sd[2 * tid + 1]};
        if (tid == k - 1 && ch == 0) *a_out = c.re;
        const bool use = tid < k && (tid == k - 1 || coef_used(c));
        const unsigned long long mask = __ballot(use);
        if (tid < 256 && (tid & 63) == 0) cnt[tid >> 6] = __popcll(mask);
        __syncthreads();
        int pos = __popcll(mask & ((1ull << (tid & 63)) - 1)), nu = 0;
        for (int w = 0; w < 4; ++w) {
            if (w < tid >> 6) pos += cnt[w];
            nu += cnt[w];
        }
        if (use) {
            sc[pos] = c;
            si[pos] = tid;
        }
        __syncthreads();
        for (int i = tid; i < N; i += kNormThreads) {
            cplx t = x[i];
#pragma unroll 4
            for (int q = 0; q < nu; ++q) {
                const cplx a = U[(int64_t)si[q] * stride + o + i], b = sc[q];
                t.re -= fma(b.re, a.re, -(b.im * a.im));
                t.im -= fma(b.im, a.re, b.re * a.im);
            }
            x[i] = t;
        }
        __syncthreads();
    }
    double acc = 0.0;
    for (int r0 = 0; r0 < N; r0 += kNormThreads) {
        const int i = r0 + tid;
        double d = 0.0;
        if (i < N) {
            double s[2 * P + 1];
            cplx y[2 * P + 1];
#pragma unroll
            for (int j = 1; j <= P; ++j) {
                s[j - 1] = i - j >= 0 ? Sd[(int64_t)j * N + max(i - j, 0)] : 0.0;
                y[j - 1] = x[max(i - j, 0)];
            }
#pragma unroll
            for (int j = 0; j <= P; ++j) {
                s[P + j] = i + j < N ? Sd[(int64_t)j * N + i] : 0.0;
                y[P + j] = x[min(i + j, N - 1)];
            }
            cplx t = {0.0, 0.0};
#pragma unroll
            for (int j = 0; j <= 2 * P; ++j) t = band_fma(s[j], y[j], t);
            d = fma(t.re, y[P].re, t.im * y[P].im);
        }
        sd[tid] = d;
        __syncthreads();
        if (tid < kNormSums)
#pragma unroll
            for (int q = 0; q < kNormThreads; q += kNormSums) acc += sd[q + tid];
        __syncthreads();
    }
    if (tid < kNormSums) sd[tid] = acc;
    __syncthreads();
    if (tid >= 64) return;
    const double s = half_sum(sd);
    if (tid == 0) npart[ch] = s;
}

__global__ __launch_bounds__(256) void k_combine(const cplx* __restrict__ U, int64_t stride, int k,
                                                 const cplx* __restrict__ c, cplx* __restrict__ w, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    cplx t = {0.0, 0.0};
#pragma unroll 4
    for (int i = 0; i < k; ++i) {
        const cplx a = U[(int64_t)i * stride + e], b = c[i];
        t.re += fma(a.re, b.re, -(a.im * b.im));
        t.im += fma(b.re, a.im, a.re * b.im);
    }
    w[e] = t;
}

// ---------------------------------------------------------------------------
// x = S^-1 v, S = C C^T (operator_sc::inverse_sub, operators/1e.hpp:1247-1251),
// partitioned as the CN solves (qpc_solve.h) with
//   forward   y_i = d_i (v_i - sum_{j=1..P} C(i,i-j) y_{i-j})
//   backward  x_i = d_i y_i - sum_{k=1..P} C(i+k,i) d_i x_{i+k},  d_i = 1 / C(i,i)
// each sum from its nearest term on.  The state a partition hands on is its
// last (first) P values; the carry looks kPKS partitions back.
//
// A row is a chain of P + 1 dependent operations, 24 rows four times; what
// bounds the launch is that chain and the loads before it.  A partition has two
// lanes of the first wave, one for the real and one for the imaginary parts (the
// tables are real), which hold its rows in registers; all waves bring rows and
// coefficients into LDS, one access each, and run the carries, a row of the
// transfer matrix each.  A work-group holds 32 partitions (the coefficients of
// both directions fill the LDS); longer channels are cut into segments with
// kPKS partitions on either side, which changes no bit.  12 channels of N = 600
// take 10.5 us, 81 of N = 3000 30.4 (all coefficients in registers instead, two
// waves of 64 partitions: 34.4 and 30.1, the waves too few to load with).
constexpr int kSParts = 32;  // partitions per work-group
constexpr int kSWaves = 8;
struct alignas(16) dbl2 {
    double x, y;
};
// Units of two coefficients: C(i,i-1) .. C(i,i-P), d_i forward, C(i+1,i) d_i ..
// C(i+P,i) d_i, d_i backward; unit u of row s and direction dir of partition g at
// ((s * 2 + dir) * real_units(P) + u) * 64 NG + g.  Entry (r, c) of a transfer
// matrix at (dir * P^2 + r * P + c) * 64 NG + g.
template <int P>
__global__ __launch_bounds__(kLane) void k_ssolve_tab(const double* __restrict__ c, dbl2* __restrict__ tab, int N,
                                                      int NP, int G) {
    constexpr int ne = P + 1, UN = real_units(P);
    const int g = blockIdx.x * kLane + threadIdx.x, s = blockIdx.y;
    if (g >= NP) return;
    const int i = g * kPM + s;
    double o[2][2 * UN] = {};  // identity padding rows
    o[0][P] = o[1][P] = 1.0;
    if (i < N) {
        const double d = 1.0 / c[(int64_t)i * ne];
        o[0][P] = o[1][P] = d;
#pragma unroll
        for (int j = 1; j <= P; ++j) {
            if (i - j >= 0) o[0][j - 1] = c[(int64_t)(i - j) * ne + j];
            if (i + j < N) o[1][j - 1] = c[(int64_t)i * ne + j] * d;
        }
    }
#pragma unroll
    for (int dir = 0; dir < 2; ++dir)
#pragma unroll
        for (int u = 0; u < UN; ++u)
            tab[(int64_t)((s * 2 + dir) * UN + u) * G + g] = dbl2{o[dir][2 * u], o[dir][2 * u + 1]};
}
// the unit responses of the state through a partition's rows, a lane per (partition, direction)
template <int P>
__global__ __launch_bounds__(kLane) void k_ssolve_trf(const dbl2* __restrict__ tab, double* __restrict__ trf, int NP,
                                                      int G) {
    constexpr int UN = real_units(P);
    const int g = blockIdx.x * kLane + threadIdx.x, dir = blockIdx.y;
    if (g >= NP) return;
    double H[P][P];  // H[q][c]: state entry q of the response to unit vector c
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int c = 0; c < P; ++c) H[q][c] = q == c ? 1.0 : 0.0;
#pragma unroll 1
    for (int ss = 0; ss < kPM; ++ss) {
        const int s = dir ? kPM - 1 - ss : ss;
        double f[2 * UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const dbl2 t = tab[(int64_t)((s * 2 + dir) * UN + u) * G + g];
            f[2 * u] = t.x;
            f[2 * u + 1] = t.y;
        }
        const double d = dir ? 1.0 : f[P];  // (backward d_i scales the row itself only)
#pragma unroll
        for (int c = 0; c < P; ++c) {
            double a = 0.0;
#pragma unroll
            for (int q = 0; q < P; ++q) a = fma(-f[q], H[q][c], a);
#pragma unroll
            for (int q = P - 1; q > 0; --q) H[q][c] = H[q - 1][c];
            H[0][c] = d * a;
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int c = 0; c < P; ++c) trf[(int64_t)(dir * P * P + q * P + c) * G + g] = H[q][c];
}

template <int P>
__global__ __launch_bounds__(kSWaves * 64) void k_ssolve(const dbl2* __restrict__ tab, const double* __restrict__ trf,
                                                         const cplx* __restrict__ vin, cplx* __restrict__ xout, int N,
                                                         int NP, int G, int SN) {
    constexpr int UN = real_units(P), NT = kSWaves * 64, NL = 2 * kSParts;
    constexpr int NU = kPM * 2 * UN * kSParts / NT, NR = (kPM * kSParts + NT - 1) / NT;  // units and rows per thread
    static_assert(P <= kSWaves && kPM * 2 * UN * kSParts % NT == 0 && NL == 64, "one wave of lanes, a row per wave");
    __shared__ dbl2 sC[kPM * 2 * UN][kSParts];  // coefficients of the staged partitions
    __shared__ dbl2 sv[kPM][kSParts + 1];       // the rows v, x
    __shared__ double sS[2][P][NL + 2];         // states, two zeros after the lanes' for the neighbour that does not exist
    const int ch = blockIdx.y, seg = blockIdx.x, tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64), ln = tid & 63, q = ln >> 1, c = ln & 1;
    const int k0 = seg * SN, k1 = min(NP, k0 + SN);             // owned partitions [k0, k1)
    const int ga = max(0, k0 - kPKS), gb = min(NP, k1 + kPKS);  // staged partitions [ga, gb)
    const int n = gb - ga, r0 = ga * kPM, nrow = n * kPM, nv = min(nrow, N - r0);
    const cplx* v = vin + (int64_t)ch * N + r0;
    // (slots past the staged partitions repeat the last; they are not used)
    cplx vr[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) vr[k] = v[min(tid + k * NT, nv - 1)];
    dbl2 cr[NU];
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const int e = tid + k * NT;
        cr[k] = tab[(int64_t)(e / kSParts) * G + min(ga + e % kSParts, gb - 1)];
    }
    double t[2][P];  // row w of this slot's transfer matrices
#pragma unroll
    for (int dir = 0; dir < 2; ++dir)
#pragma unroll
        for (int j = 0; j < P; ++j) t[dir][j] = trf[(int64_t)((dir * P + min(w, P - 1)) * P + j) * G + min(ga + q, gb - 1)];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int i = tid + k * NT;
        if (i < kPM * kSParts) sv[i % kPM][i / kPM] = i < nv ? dbl2{vr[k].re, vr[k].im} : dbl2{0.0, 0.0};
    }
#pragma unroll
    for (int k = 0; k < NU; ++k) sC[(tid + k * NT) / kSParts][(tid + k * NT) % kSParts] = cr[k];
    if (tid < 4 * P) sS[tid / (2 * P)][tid / 2 % P][NL + tid % 2] = 0.0;
    __syncthreads();
    double y[kPM], h[P];
    double* row = &sv[0][0].x + ln;  // this lane's part of its partition's first row
    constexpr int rstep = 2 * (kSParts + 1);
    auto coefs = [&](double (&f)[2 * UN], int s, int dir) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const dbl2 a = sC[(s * 2 + dir) * UN + u][q];
            f[2 * u] = a.x;
            f[2 * u + 1] = a.y;
        }
    };
    if (w == 0)
#pragma unroll
        for (int s = 0; s < kPM; ++s) y[s] = row[s * rstep];
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
#pragma unroll
        for (int j = 0; j < P; ++j) h[j] = 0.0;
#pragma unroll 1
        for (int pass = 0;; ++pass) {
            if (w == 0) {
#pragma unroll
                for (int ss = 0; ss < kPM; ++ss) {
                    const int s = dir ? kPM - 1 - ss : ss;
                    double f[2 * UN];
                    coefs(f, s, dir);
                    double a = dir ? fma(f[P], y[s], -(f[0] * h[0])) : fma(-f[0], h[0], y[s]);
#pragma unroll
                    for (int j = 1; j < P; ++j) a = fma(-f[j], h[j], a);
                    if (!dir) a = f[P] * a;
#pragma unroll
                    for (int j = P - 1; j > 0; --j) h[j] = h[j - 1];
                    h[0] = a;
                    y[s] = pass ? a : y[s];
                }
            }
            if (pass) break;
            // the incoming state from the pass-A end states h: s_g <- h_g + T_g
            // s_{g-1} (g+1 backward), kPKS - 1 times from s = h; wave w has row w
            const int nb = dir == 0 ? (q > 0 ? ln - 2 : NL + c) : (q + 1 < n ? ln + 2 : NL + c);
            if (w == 0)
#pragma unroll
                for (int r = 0; r < P; ++r) sS[0][r][ln] = h[r];
            __syncthreads();
            const double e = sS[0][min(w, P - 1)][ln];
#pragma unroll 1
            for (int k = 1; k < kPKS; ++k) {
                if (w < P) {
                    double in[P], a = e;
#pragma unroll
                    for (int j = 0; j < P; ++j) in[j] = sS[(k - 1) & 1][j][nb];
#pragma unroll
                    for (int j = 0; j < P; ++j) a = fma(t[dir][j], in[j], a);
                    sS[k & 1][w][ln] = a;
                }
                __syncthreads();
            }
            if (w == 0)
#pragma unroll
                for (int r = 0; r < P; ++r) h[r] = sS[(kPKS - 1) & 1][r][nb];
        }
    }
    if (w == 0)
#pragma unroll
        for (int s = 0; s < kPM; ++s) row[s * rstep] = y[s];
    __syncthreads();
    cplx* x = xout + (int64_t)ch * N + r0;
    const int i0 = (k0 - ga) * kPM, i1 = min((k1 - ga) * kPM, nv);
    for (int i = i0 + tid; i < i1; i += NT) x[i] = cplx{sv[i % kPM][i / kPM].x, sv[i % kPM][i / kPM].y};
}

}  // namespace

void launch_hmul(hipStream_t s, const double* Hd, const double* Fd, const double* Gd, const double* y10,
                 const double* q10, double az, int M, int L, int m0, int N, int p, const cplx* v, const double* npart,
                 int first, double* b_out, cplx* u, cplx* t) {
    const dim3 grid((N + kTile - 1) / kTile, M * L);
    if (p == 8)
        hipLaunchKernelGGL(k_hmul<8>, grid, dim3(kTile), 0, s, Hd, Fd, Gd, y10, q10, az, L, m0, N, v, npart, M * L,
                           first, b_out, u, t);
    else
        hipLaunchKernelGGL(k_hmul<7>, grid, dim3(kTile), 0, s, Hd, Fd, Gd, y10, q10, az, L, m0, N, v, npart, M * L,
                           first, b_out, u, t);
}
void launch_norm_final(hipStream_t s, int nch, const double* npart, double* b_out) {
    hipLaunchKernelGGL(k_norm_final, dim3(1), dim3(64), 0, s, npart, nch, b_out);
}
void launch_dots(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* v, int64_t n, cplx* part) {
    hipLaunchKernelGGL(k_dots, dim3(kDotBlocks, k), dim3(256), 0, s, U, stride, v, n, part);
}
void launch_axpy_norm(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* part, double* a_out,
                      const double* Sd, cplx* v, int N, int nch, int p, double* npart) {
    const dim3 block(kNormThreads);
    if (p == 8)
        hipLaunchKernelGGL(k_axpy_norm<8>, dim3(nch), block, 0, s, U, stride, k, (const double*)part, a_out, Sd, v, N,
                           npart);
    else
        hipLaunchKernelGGL(k_axpy_norm<7>, dim3(nch), block, 0, s, U, stride, k, (const double*)part, a_out, Sd, v, N,
                           npart);
}
void launch_combine(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* c, cplx* w, int64_t n) {
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, U, stride, k, c, w, n);
}

int64_t ssolve_tab_elems(const Geom& geo) { return (int64_t)geo.NG * kLane * kPM * 4 * real_units(geo.hw); }
int64_t ssolve_trf_elems(const Geom& geo) { return (int64_t)geo.NG * kLane * 2 * geo.hw * geo.hw; }
template <int P>
static void ssolve_tables(hipStream_t s, const double* chol, double* tab, double* trf, const Geom& geo) {
    const int G = geo.NG * kLane;
    hipLaunchKernelGGL(k_ssolve_tab<P>, dim3(geo.NG, kPM), dim3(kLane), 0, s, chol, (dbl2*)tab, geo.N, geo.P, G);
    hipLaunchKernelGGL(k_ssolve_trf<P>, dim3(geo.NG, 2), dim3(kLane), 0, s, (const dbl2*)tab, trf, geo.P, G);
}
void launch_ssolve_tables(hipStream_t s, const double* chol, double* tab, double* trf, const Geom& geo) {
    if (geo.hw == 8) ssolve_tables<8>(s, chol, tab, trf, geo);
    else ssolve_tables<7>(s, chol, tab, trf, geo);
}
void launch_ssolve(hipStream_t s, const double* tab, const double* trf, const cplx* v, cplx* x, int nch,
                   const Geom& geo) {
    constexpr int smax = kSParts - 2 * kPKS;
    const int ns = geo.P <= kSParts ? 1 : (geo.P + smax - 1) / smax;
    const int SN = (geo.P + ns - 1) / ns, nseg = (geo.P + SN - 1) / SN, G = geo.NG * kLane;
    const dim3 grid(nseg, nch), block(kSWaves * 64);
    if (geo.hw == 8)
        hipLaunchKernelGGL(k_ssolve<8>, grid, block, 0, s, (const dbl2*)tab, trf, v, x, geo.N, geo.P, G, SN);
    else
        hipLaunchKernelGGL(k_ssolve<7>, grid, block, 0, s, (const dbl2*)tab, trf, v, x, geo.N, geo.P, G, SN);
}

}  // namespace qpc
