// qpc_krylov.hip -- device pieces of the Krylov propagator (gfx950).
//
// A Lanczos vector of a small grid is bound by what lies between its kernels,
// not by them: two host round trips for its products and norm, with their
// copies, took half of its 119 us (N = 600, L = 12).  The chain therefore
// stays on the device: the products of k_dots are summed where k_axpy_norm
// uses them, the norm it leaves in partial sums is finished by the next
// vector's k_hmul, which also normalises the vector, and the tridiagonal goes
// to host memory that the device writes.
// A vector now takes 37 us, 25 of them in its four kernels: k_hmul 4.9 us (was
// 11.3), k_dots 4.2, the solve 8.6 (21), k_axpy_norm 6.8 (6.2 with 8.6 for the
// norm and 2.2 for the scaling).
#include "qpc_krylov.h"

#include <algorithm>

namespace qpc {
namespace {

constexpr int kTile = 128;      // rows per work-group of k_hmul
constexpr int kAxpyTile = 256;  // rows per tile of k_axpy_norm

__device__ inline cplx times_i(cplx z, double a) { return {-a * z.im, a * z.re}; }  // i a z

// sum over the work-group of NT threads, in a fixed order
template <int NT>
__device__ inline double group_sum(double v) {
    __shared__ double s[NT];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int st = NT / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
        __syncthreads();
    }
    const double r = s[0];
    __syncthreads();
    return r;
}
template <int NT>
__device__ inline double norm_sum(const double* __restrict__ part, int np) {
    double a = 0.0;
    for (int i = threadIdx.x; i < np; i += NT) a += part[i];
    return group_sum<NT>(a);
}
// b_k from the squared norm (orthogonalize_ip, la_1e.hpp:195-240: below 1e-13
// the subspace ends; the first vector's is always used)
__device__ inline double norm_of(double s, int first) { return !first && s < 1e-13 ? 0.0 : sqrt(s); }

// u = v / |v|, t = H(az) u over every channel: H_l u plus, from the channels
// l - 1 and l + 1 of u, i az F y and i az G w with y = q(l-1) u(l-1) - q(l) u(l+1)
// and w = -y(l-1) u(l-1) - y(l) u(l+1) (three banded products instead of
// five).  A row's operands are 3 (2 P + 1) band entries, all requested before
// their first use, and u, y, w from LDS.
template <int P>
__global__ __launch_bounds__(kTile) void k_hmul(const double* __restrict__ Hd, const double* __restrict__ Fd,
                                                const double* __restrict__ Gd, const double* __restrict__ y10,
                                                const double* __restrict__ q10, double az, int L, int m0, int N,
                                                const cplx* __restrict__ v, const double* __restrict__ npart, int np,
                                                int first, double* b_out, cplx* __restrict__ u, cplx* __restrict__ t) {
    constexpr int NX = kTile + 2 * P;
    __shared__ cplx sx[NX], sy[NX], sw[NX];
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
    }
#pragma unroll
    for (int j = 1; j <= P; ++j) {
        const int64_t o = (int64_t)j * N + max(ic - j, 0);
        hl[j - 1] = H[o];
        fl[j - 1] = Fd[o];
        gl[j - 1] = Gd[o];
    }
    const double qm = il > 0 ? q10[ch - 1] : 0.0, ym = il > 0 ? y10[ch - 1] : 0.0;
    const double qp = il < L - 1 ? q10[ch] : 0.0, yp = il < L - 1 ? y10[ch] : 0.0;
    const cplx* x = v + (int64_t)ch * N;
    const cplx zero = {0.0, 0.0};
    cplx xc[2], xm[2], xp[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = r0 - P + tid + k * kTile;
        const bool in = r >= 0 && r < N && tid + k * kTile < NX;
        const int rc = in ? r : 0;
        xc[k] = x[rc];
        xm[k] = x[rc - (il > 0 ? N : 0)];
        xp[k] = x[rc + (il < L - 1 ? N : 0)];
        if (!in) xc[k] = zero;
        if (!in || il == 0) xm[k] = zero;
        if (!in || il == L - 1) xp[k] = zero;
    }
    const double nk = norm_of(norm_sum<kTile>(npart, np), first);
    if (blockIdx.x == 0 && ch == 0 && tid == 0) *b_out = nk;
    const double inv = nk == 0.0 ? 0.0 : 1.0 / nk;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int e = tid + k * kTile;
        const cplx a = xc[k] * inv, bm = xm[k] * inv, bp = xp[k] * inv;
        if (e < NX) {
            sx[e] = a;
            sy[e] = bm * qm - bp * qp;
            sw[e] = zero - bm * ym - bp * yp;
        }
    }
    __syncthreads();
    if (i >= N) return;
    cplx h = zero, f = zero, g = zero;
#pragma unroll
    for (int j = P; j >= 1; --j) {
        h += hl[j - 1] * sx[tid + P - j];
        f += fl[j - 1] * sy[tid + P - j];
        g -= gl[j - 1] * sw[tid + P - j];
    }
#pragma unroll
    for (int k = 0; k <= P; ++k) {
        h += hu[k] * sx[tid + P + k];
        f += fu[k] * sy[tid + P + k];
        g += gu[k] * sw[tid + P + k];
    }
    u[(int64_t)ch * N + i] = sx[tid + P];
    t[(int64_t)ch * N + i] = h + times_i(f, az) + times_i(g, az);
}

__global__ __launch_bounds__(kTile) void k_norm_final(const double* __restrict__ npart, int np, double* b_out) {
    const double s = norm_sum<kTile>(npart, np);
    if (threadIdx.x == 0) *b_out = norm_of(s, 0);
}

__global__ __launch_bounds__(256) void k_dots(const cplx* __restrict__ U, int64_t stride, const cplx* __restrict__ v,
                                              int64_t n, cplx* __restrict__ part) {
    __shared__ double sre[256], sim[256];
    const int b = blockIdx.x, vi = blockIdx.y, nb = gridDim.x;
    const cplx* u = U + (int64_t)vi * stride;
    const int64_t chunk = (n + nb - 1) / nb;
    const int64_t e0 = (int64_t)b * chunk, e1 = e0 + chunk < n ? e0 + chunk : n;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) {
        const cplx a = u[e], c = v[e];
        re += a.re * c.re + a.im * c.im;
        im += a.re * c.im - a.im * c.re;
    }
    sre[threadIdx.x] = re;
    sim[threadIdx.x] = im;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            sre[threadIdx.x] += sre[threadIdx.x + st];
            sim[threadIdx.x] += sim[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(int64_t)vi * nb + b] = cplx{sre[0], sim[0]};
}

// v -= sum_{i<k} c_i U_i with c_i the sum of k_dots' nb partials, left out
// where |c_i|^2 <= 4e-27 (the last is always used); a_out = Re c_{k-1}; and the
// partial sums of <v|S|v>, one per work-group.  A work-group computes its tile
// and the P rows after it (k = 0: only the norm of v).
template <int P>
__global__ __launch_bounds__(kAxpyTile) void k_axpy_norm(const cplx* __restrict__ U, int64_t stride, int k,
                                                         const cplx* __restrict__ part, int nb, double* a_out,
                                                         const double* __restrict__ Sd, const cplx* __restrict__ vin,
                                                         cplx* __restrict__ vout, int N, int nch,
                                                         double* __restrict__ npart) {
    constexpr int NT = kAxpyTile;
    __shared__ cplx sc[256], sv[NT + P];
    __shared__ int si[256], cnt[NT / 64];
    const int tid = threadIdx.x;
    // the coefficients in use, compacted in order (k <= 256)
    cplx c = {0.0, 0.0};
    if (tid < k) {
#pragma unroll 8
        for (int q = 0; q < nb; ++q) c += part[(int64_t)tid * nb + q];
        if (tid == k - 1 && blockIdx.x == 0) *a_out = c.re;
    }
    const bool use = tid < k && (tid == k - 1 || c.re * c.re + c.im * c.im > 4e-27);
    const unsigned long long mask = __ballot(use);
    if ((tid & 63) == 0) cnt[tid >> 6] = __popcll(mask);
    __syncthreads();
    int pos = __popcll(mask & ((1ull << (tid & 63)) - 1)), nu = 0;
    for (int w = 0; w < NT / 64; ++w) {
        if (w < tid >> 6) pos += cnt[w];
        nu += cnt[w];
    }
    if (use) {
        sc[pos] = c;
        si[pos] = tid;
    }
    __syncthreads();
    const int tpc = (N + NT - 1) / NT;  // tiles per channel
    const int64_t tiles = (int64_t)tpc * nch;
    double acc = 0.0;
    for (int64_t tl = blockIdx.x; tl < tiles; tl += gridDim.x) {
        const int ch = (int)(tl / tpc), r0 = (int)(tl % tpc) * NT;
        const int i = r0 + tid;
        double s[P + 1];
#pragma unroll
        for (int j = 0; j <= P; ++j) s[j] = Sd[(int64_t)j * N + min(i, N - 1)];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = tid + h * NT, r = r0 + e;
            if (e >= NT + P) continue;
            cplx t = {0.0, 0.0};
            if (r < N) {
                const int64_t o = (int64_t)ch * N + r;
                t = vin[o];
#pragma unroll 4
                for (int q = 0; q < nu; ++q) t -= U[(int64_t)si[q] * stride + o] * sc[q];
                if (h == 0 && k > 0) vout[o] = t;
            }
            sv[e] = t;
        }
        __syncthreads();
        if (i < N) {
            // x_i* (S x)_i with the pairs (i, i + j) once, doubled
            const cplx x = sv[tid];
            double d = 0.0;
#pragma unroll
            for (int j = P; j >= 1; --j) {
                const cplx y = sv[tid + j];
                d += s[j] * (x.re * y.re + x.im * y.im);
            }
            acc += 2.0 * d + s[0] * (x.re * x.re + x.im * x.im);
        }
        __syncthreads();
    }
    const double sum = group_sum<NT>(acc);
    if (tid == 0) npart[blockIdx.x] = sum;
}

__global__ __launch_bounds__(256) void k_combine(const cplx* __restrict__ U, int64_t stride, int k,
                                                 const cplx* __restrict__ c, cplx* __restrict__ w, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    cplx t = U[e] * c[0];
#pragma unroll 4
    for (int i = 1; i < k; ++i) t += U[(int64_t)i * stride + e] * c[i];
    w[e] = t;
}

}  // namespace

int dot_blocks(int64_t n) { return (int)std::min<int64_t>(kDotBlocks, std::max<int64_t>(1, (n + 1023) / 1024)); }

int norm_blocks(int N, int nch) {
    return (int)std::min<int64_t>(kNormBlocks, (int64_t)((N + kAxpyTile - 1) / kAxpyTile) * nch);
}

void launch_hmul(hipStream_t s, const double* Hd, const double* Fd, const double* Gd, const double* y10,
                 const double* q10, double az, int M, int L, int m0, int N, int p, const cplx* v, const double* npart,
                 int first, double* b_out, cplx* u, cplx* t) {
    const dim3 grid((N + kTile - 1) / kTile, M * L);
    const int np = norm_blocks(N, M * L);
    if (p == 8)
        hipLaunchKernelGGL(k_hmul<8>, grid, dim3(kTile), 0, s, Hd, Fd, Gd, y10, q10, az, L, m0, N, v, npart, np, first,
                           b_out, u, t);
    else
        hipLaunchKernelGGL(k_hmul<7>, grid, dim3(kTile), 0, s, Hd, Fd, Gd, y10, q10, az, L, m0, N, v, npart, np, first,
                           b_out, u, t);
}
void launch_norm_final(hipStream_t s, int N, int nch, const double* npart, double* b_out) {
    hipLaunchKernelGGL(k_norm_final, dim3(1), dim3(kTile), 0, s, npart, norm_blocks(N, nch), b_out);
}
void launch_dots(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* v, int64_t n, cplx* part) {
    hipLaunchKernelGGL(k_dots, dim3(dot_blocks(n), k), dim3(256), 0, s, U, stride, v, n, part);
}
void launch_axpy_norm(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* part, double* a_out,
                      const double* Sd, const cplx* vin, cplx* vout, int N, int nch, int p, double* npart) {
    const dim3 grid(norm_blocks(N, nch));
    const int nb = dot_blocks((int64_t)N * nch);
    if (p == 8)
        hipLaunchKernelGGL(k_axpy_norm<8>, grid, dim3(kAxpyTile), 0, s, U, stride, k, part, nb, a_out, Sd, vin, vout, N,
                           nch, npart);
    else
        hipLaunchKernelGGL(k_axpy_norm<7>, grid, dim3(kAxpyTile), 0, s, U, stride, k, part, nb, a_out, Sd, vin, vout, N,
                           nch, npart);
}
void launch_combine(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* c, cplx* w, int64_t n) {
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, U, stride, k, c, w, n);
}

}  // namespace qpc
