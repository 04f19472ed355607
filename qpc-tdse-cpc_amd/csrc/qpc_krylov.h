// qpc_krylov.h -- device pieces of the Krylov (S-orthogonal Lanczos) propagator,
// propagator_arnoldi with propagator_hc_vgwz::multiply (la_1e.hpp:90-335, 480-497).
#pragma once
#include "qpc_common.h"

namespace qpc {

constexpr int kDotBlocks = 128;    // most partial sums per inner product (dot_blocks)
constexpr int kNormBlocks = 1024;  // most partial sums of a squared S-norm (norm_blocks)

// u = v / |v|_S with |v|_S^2 the sum of npart (u = 0 where it is below 1e-13,
// unless first), *b_out = |v|_S (0 there), and t = H(az) u over every channel
// (la_1e.hpp:480-497): H_l per channel and the l -> l+-1 couplings
// +i az q(l-1) F - i az y(l-1) G  (from l-1) and -i az y(l) G - i az q(l) F
// (from l+1); F = <Bi|1/r|Bj> symmetric, G = <Bi|d/dr Bj> antisymmetric; all
// bands diagonal-major (D[j*N+i] = A(i,i+j)), H per l at Hd + l*(p+1)*N; p is
// n_rank (7 or 8).
void launch_hmul(hipStream_t s, const double* Hd, const double* Fd, const double* Gd, const double* y10,
                 const double* q10, double az, int M, int L, int m0, int N, int p, const cplx* v, const double* npart,
                 int first, double* b_out, cplx* u, cplx* t);
// *b_out alone
void launch_norm_final(hipStream_t s, int N, int nch, const double* npart, double* b_out);
// partial sums of conj(U_i) . v, i < k, for launch_axpy_norm
void launch_dots(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* v, int64_t n, cplx* part);
// vout = vin - sum_{i<k} c_i U_i with c_i summed from part (terms of |c_i|^2 <=
// 4e-27 left out but for the last), *a_out = Re c_{k-1}, npart = partial sums
// of vout's squared S-norm (k = 0: of vin's, and nothing else); vin and vout differ
void launch_axpy_norm(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* part, double* a_out,
                      const double* Sd, const cplx* vin, cplx* vout, int N, int nch, int p, double* npart);
// w = sum_{i<k} c[i] U_i
void launch_combine(hipStream_t s, const cplx* U, int64_t stride, int k, const cplx* c, cplx* w, int64_t n);

}  // namespace qpc
