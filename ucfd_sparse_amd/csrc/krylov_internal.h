// Internal interface between the Krylov host code (krylov_api.cpp) and its
// kernels (krylov_kernels.hip).  Not installed.
#pragma once

#include <stdint.h>

#include "ucfd_internal.h"

// Deterministic reductions: a kernel writes one partial per block (and per
// reduced quantity), a second kernel sums them in a fixed order.
constexpr int KRY_BLOCK = 256;

// y = alpha*A*x + beta*y for a BSR matrix (row-major blk x blk blocks,
// vectors stored x[row*blk + r]); one thread per block row, the operation
// order of src/krylov/matrix/sparsemat.c:57-101.
UCFD_HIDDEN int kry_spmv_bsr(hipStream_t s, int bn, int blk, const int *rowptr, const int *colidx,
                             const double *values, double alpha, const double *x, double beta,
                             double *y, int *flag);
// Scalar CSR form (sparsemat.c:10-29).  Both raise UCFD_KFLAG_INDEX for a
// column index outside the matrix (the entry is skipped).
UCFD_HIDDEN int kry_spmv_csr(hipStream_t s, int n, const int *rowptr, const int *colidx,
                             const double *values, double alpha, const double *x, double beta,
                             double *y, int *flag);

// diagvalues[i] = LU(values[diagslots[i]]) (FP64, Doolittle without pivoting);
// raises UCFD_KFLAG_PIVOT on a zero pivot.  vals32 (nullable): FP32 copy of
// every block for the mixed-precision apply.
UCFD_HIDDEN int kry_bsgs_prepare(hipStream_t s, int bn, int blk, int64_t nnz, const int *diagslots,
                                 const double *values, double *diagvalues, float *vals32,
                                 int *flag);

// One level of the in-place ILU(0) factorisation (rows base..base+cnt-1, or
// order[base..]): scalar != 0 is ILU(0) of a CSR matrix (blk 1, ilu.c:4-48),
// else block ILU(0) (bilu.c:5-65).  diagvalues[i] gets row i's factored
// diagonal block (scalar: its pivot); raises UCFD_KFLAG_PIVOT on a zero pivot.
// rows != 0 (block form): no lower slot of a row refers to the row itself,
// which lets the lanes of a wave share a row's block operations.
UCFD_HIDDEN int kry_ilu_factor(hipStream_t s, int scalar, int rows, int blk, int base, int cnt,
                               const int *order, const int *rowptr, const int *colidx,
                               const int *diagslots, double *values, double *diagvalues,
                               int *flag);

// Sweep kinds of kry_bsgs_sweep64
enum { KRY_SW_LUSGS = 0, KRY_SW_BILU = 1, KRY_SW_ILU = 2 };

// One sweep over rows base..base+cnt-1 (or order[base..base+cnt-1] when
// order != NULL), in place on b.  KRY_SW_LUSGS: lower x_i = D_i^-1 (b_i -
// sum_{j<diag} A_ij x_j), upper x_i -= D_i^-1 sum_{j>diag} A_ij x_j.
// KRY_SW_BILU (factored values): lower x_i = b_i - sum_{j<diag} L_ij x_j,
// upper x_i = U_ii^-1 (x_i - sum_{j>diag} U_ij x_j) with diagvalues the
// factored U_ii.  KRY_SW_ILU: the scalar form (blk 1), dividing by the pivot.
// empty: no row of the (contiguous) level has a block in this direction.  join (a
// lower sweep of a contiguous level, blk > 1): each row's update of the upper sweep
// follows at once, for rows with no block above the diagonal.
UCFD_HIDDEN int kry_bsgs_sweep64(hipStream_t s, int kind, int upper, int blk, int base, int cnt,
                                 const int *order, const int *rowptr, const int *colidx,
                                 const int *diagslots, const double *values,
                                 const double *diagvalues, double *b, bool empty, bool join);
// Mixed form: block products in FP32 on FP32 values and an FP32 work vector
// x32, the diagonal solve in FP64.  lower reads the right-hand side b (FP64)
// and writes x32; upper updates x32 and writes the final value to b (FP64).
UCFD_HIDDEN int kry_bsgs_sweep32(hipStream_t s, int upper, int blk, int base, int cnt,
                                 const int *order, const int *rowptr, const int *colidx,
                                 const int *diagslots, const float *vals32,
                                 const double *diagvalues, float *x32, double *b, bool empty,
                                 bool join);

// Scalars posted to the host by the kernel that forms them: values at out (the
// device address of pinned memory), then seq at word (0: not yet the last).
// out NULL: nothing posted.
struct KryPost {
    double *out = nullptr;
    unsigned long long *word = nullptr, seq = 0;
};
struct KryCoef {
    double v[64];
};

// BLAS-1/2 on device vectors.  A reduction leaves its partials, or the one sum
// where they would be many, in row q at part + q*KRY_MAXPART; the kernel that
// uses it (over vectors of the same length) sums the row in a fixed order.
enum { KRY_MAXPART = 1024 };
// x.y: partials, and with out also the sum (device, posted)
UCFD_HIDDEN int kry_dot(hipStream_t s, int64_t n, const double *x, const double *y, double *part,
                        double *out, const KryPost &h = KryPost());
UCFD_HIDDEN int kry_axpy(hipStream_t s, int64_t n, double a, const double *x, double *y);
UCFD_HIDDEN int kry_axpby(hipStream_t s, int64_t n, double a, const double *x, double b,
                          double *y);  // y = a x + b y
// dst = src/sqrt(the sum of the partials nsq_part, posted); the same values also
// into dst2 when given
UCFD_HIDDEN int kry_scale_by_inv_sqrt(hipStream_t s, int64_t n, const double *src,
                                      const double *nsq_part, double *dst, double *dst2,
                                      const KryPost &h = KryPost());
// partials of h[j] = sum_i V[j*ldv + i] w[i], j < k (k <= 64)
UCFD_HIDDEN int kry_gemvt(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv,
                          const double *w, double *part);
// w[i] += alpha * sum_j V[j*ldv + i] h[j], h the sums of the partials hpart
// (posted); with part also the partials of sum_i w_new[i]^2.  part is not hpart.
UCFD_HIDDEN int kry_gemv(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv,
                         double alpha, const double *hpart, double *w, double *part,
                         const KryPost &h = KryPost());
// kry_gemv (no norm) followed by kry_gemvt on the updated w, in one pass over
// V when k <= 32.  part is not hpart.
UCFD_HIDDEN int kry_gemv_gemvt(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv,
                               double alpha, const double *hpart, double *w, double *part,
                               const KryPost &h = KryPost());
// x += V y
UCFD_HIDDEN int kry_gemv_y(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv,
                           const KryCoef &y, double *x);
// BiCGSTAB fused reduction (bicgstab.c:5-22): partials of (rt.s, rt.t, t.s, t.t,
// s.s) in rows 0..4
UCFD_HIDDEN int kry_dot5(hipStream_t s, int64_t n, const double *rt, const double *sv,
                         const double *t, double *part);
// p = r + beta*(p - omega*v); pt = p
UCFD_HIDDEN int kry_bicg_p(hipStream_t s, int64_t n, double beta, double omega, const double *r,
                           const double *v, double *p, double *pt);
// s = r - alpha*v; shat = s, with alpha = rho / pi, pi the sum of pi_part
UCFD_HIDDEN int kry_bicg_s(hipStream_t s, int64_t n, double rho, const double *pi_part,
                           const double *r, const double *v, double *sv, double *shat);
// b = (float)a
UCFD_HIDDEN int kry_cast32(hipStream_t s, int64_t n, const double *a, float *b);
// pi and the five dots from their partials (posted as dots 0..4, pi), then
// x += alpha*pt + omega*shat; r = s - omega*t with alpha = rho/pi, omega =
// t.s/t.t; |pi| < 1e-30 leaves x and r alone
UCFD_HIDDEN int kry_bicg_xr(hipStream_t s, int64_t n, double rho, const double *pi_part,
                            const double *dots, const double *pt, const double *shat,
                            const double *sv, const double *t, double *x, double *r,
                            const KryPost &h);
UCFD_HIDDEN int kry_copy(hipStream_t s, int64_t n, const double *x, double *y);
UCFD_HIDDEN int kry_fill(hipStream_t s, int64_t n, double v, double *y);
