// qpc_krylov.h -- device pieces of the Krylov propagator (propagator_arnoldi,
// propagator/la_1e.hpp:64-338, 428-558).
//
// The sums of the chain have one order, stated at each kernel, with the fused
// multiply-adds written out: a-posteriori estimates far below the tolerance are
// rounding of these sums, and a controller's steps follow the estimates, so
// that another order moves a controlled run by up to 4e-7
// (tests/test_gpu_krylov_order.py holds the bits).
#pragma once
#include "qpc_common.h"
#include "qpc_solve.h"

namespace qpc {

constexpr int kDotBlocks = 128;  // partial sums per inner product

// u = v / |v|_S with |v|_S^2 the sum of the channels' npart (u = 0 where it is
// below 1e-13, unless first), *b_out = |v|_S (0 there), and t = H(az) u over
// every channel (la_1e.hpp:480-497): H_l per channel and the l -> l+-1
// couplings +i az q(l-1) F - i az y(l-1) G  (from l-1) and -i az y(l) G - i az
// q(l) F  (from l+1); F = <Bi|1/r|Bj> symmetric, G = <Bi|d/dr Bj>
// antisymmetric; all bands diagonal-major (D[j*N+i] = A(i,i+j)), H per l at
// Hd + l*(p+1)*N; p is n_rank (7 or 8).
void launch_hmul(hipStream_t s, const double* Hd, const double* Fd, const double* Gd, const double* y10,
                 const double* q10, double az, int M, int L, int m0, int N, int p, const cplx* v, const double* npart,
                 int first, double* b_out, cplx* u, cplx* t);
// *b_out alone
void launch_norm_final(hipStream_t s, int nch, const double* npart, double* b_out);
// partial sums of conj(U_i) . v, i < k, for launch_axpy_norm
void launch_dots(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* v, int64_t n, cplx* part);
// v -= sum_{i<k} c_i U_i with c_i summed from part (terms of |c_i|^2 <= 4e-27
// left out but for the last), *a_out = Re c_{k-1}, and npart[ch] = v's squared
// S-norm in channel ch (k = 0: the norms alone)
void launch_axpy_norm(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* part, double* a_out,
                      const double* Sd, cplx* v, int N, int nch, int p, double* npart);
// w = sum_{i<k} c[i] U_i
void launch_combine(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* c, cplx* w, int64_t n);

// x = S^-1 v for nch channels, tables from chol(S) (row-major, L(i+j,i))
int64_t ssolve_tab_elems(const Geom& geo);
int64_t ssolve_trf_elems(const Geom& geo);
void launch_ssolve_tables(hipStream_t s, const double* chol, double* tab, double* trf, const Geom& geo);
void launch_ssolve(hipStream_t s, const double* tab, const double* trf, const cplx* v, cplx* x, int nch,
                   const Geom& geo);

}  // namespace qpc
