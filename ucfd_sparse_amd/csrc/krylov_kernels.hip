// Kernels of the Krylov path: BSR / CSR SpMV, block LU-SGS (prepare, lower
// and upper sweeps in FP64 and in the mixed FP32/FP64 form), the ILU(0)
// family (level-scheduled factorisation, triangular solves), BLAS-1/2 with
// deterministic reductions, and the fused BiCGSTAB vector updates.
//
// FP64 kernels keep the operation order of the reference
// (src/krylov/matrix/sparsemat.c:57-101, src/krylov/utils/inverse.c:7-107,
// src/krylov/precon/blusgs.c:28-100, ilu.c:4-86, bilu.c:5-130, pbilu.c:5-180)
// and are compiled without FMA contraction, so SpMV, the factorisations and
// the FP64 preconditioner applies agree bit for bit with the CPU oracle.
// Reductions sum block partials in a fixed order, so every dot product is
// reproducible run to run.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "block_lu.h"
#include "error_word.h"
#include "krylov_internal.h"
#include "wave_rows.h"

namespace {

constexpr int KB = KRY_BLOCK;
constexpr int KMAXPART = KRY_MAXPART;

__device__ __forceinline__ int kxcd()
{
    const int b = blockIdx.x, nblk = gridDim.x;
    const int x = b % 8, k = b / 8, per = nblk / 8, rem = nblk % 8;
    return x*per + (x < rem ? x : rem) + k;
}

inline int nblocks(int64_t n)
{
    const int64_t b = (n + KB - 1)/KB;
    return (int)(b < 1 ? 1 : (b > KMAXPART ? KMAXPART : b));
}

// ------------------------------------------------------------------ SpMV
template <int B>
__global__ __launch_bounds__(KB) void k_spmv_bsr(int bn, const int *__restrict__ rowptr,
                                                 const int *__restrict__ colidx,
                                                 const double *__restrict__ values, double alpha,
                                                 const double *__restrict__ x, double beta,
                                                 double *__restrict__ y, int *flag)
{
    const int idx = kxcd()*KB + threadIdx.x;
    if (idx >= bn) return;
    bool bad = false;
    double arr[B];
#pragma unroll
    for (int k = 0; k < B; ++k) arr[k] = 0.0;
    const int st = rowptr[idx], ed = rowptr[idx + 1];
    for (int j = st; j < ed; ++j) {
        const int c = colidx[j];
        if ((unsigned)c >= (unsigned)bn) {
            bad = true;
            continue;
        }
        const double *blk = values + (int64_t)j*B*B;
        double xp[B];
#pragma unroll
        for (int r = 0; r < B; ++r) xp[r] = x[(int64_t)c*B + r];
#pragma unroll
        for (int r = 0; r < B; ++r) {
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < B; ++q) v += __builtin_nontemporal_load(blk + r*B + q)*xp[q];
            arr[r] += v;
        }
    }
#pragma unroll
    for (int k = 0; k < B; ++k) {
        const int64_t o = (int64_t)idx*B + k;
        y[o] = alpha*arr[k] + beta*y[o];
    }
    if (bad) ucfd::raise(flag, UCFD_KFLAG_INDEX);
}

// Block sizes 2..7: one wave per G = 64/B block rows; lane (g, r) sums scalar row
// r of block row g in the reference order (per block: v = sum_q A[r][q] x[q],
// then arr += v).  A lane reads its B values of a block, and the x row it meets,
// in the widest loads that cover them (wave_rows.h), KP blocks' loads together:
// 3 + 3 loads a 5x5 block.  Temporal loads: a block's lines serve all B lanes
// and several loads (non-temporal ones fetched them again: 89 -> 135 us).
// Against blocks staged through LDS with consecutive lanes on consecutive words
// (one scalar load per 64 values, then LDS): 64K hex rows 31.8 -> 21.5 us, 384K
// tet rows 89.6 -> 82.7, 1M 223 -> 216 (4.6 TB/s of matrix values); 4x4 blocks,
// 384K rows, 57.4 -> 49.1, 7x7 162.6 -> 155.9.  KP: a tet's whole row of five
// blocks where the registers allow it (5x5: 82.7 us with 5, 87.8 with 3; 7x7:
// 155.9 with 3, 163 with 5).
template <int B>
__global__ __launch_bounds__(64) void k_spmv_bsr_w(int bn, const int *__restrict__ rowptr,
                                                   const int *__restrict__ colidx,
                                                   const double *__restrict__ values,
                                                   double alpha, const double *__restrict__ x,
                                                   double beta, double *__restrict__ y, int *flag)
{
    constexpr int B2 = B*B, G = 64/B, KP = B <= 5 ? 5 : 3;
    const int lane = threadIdx.x, g = lane/B, r = lane%B;
    const int i = ucfd::wave_xcd_index()*G + g;
    if (g >= G || i >= bn) return;
    const int st = rowptr[i], ed = rowptr[i + 1];
    bool bad = false;
    double arr = 0.0;
    for (int j0 = st; j0 < ed; j0 += KP) {
        int c[KP];
        double a[KP][B], xv[KP][B];
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (j0 + k < ed) {
                c[k] = colidx[j0 + k];
                ucfd::ld_values<B>(values + (int64_t)(j0 + k)*B2 + r*B, a[k]);
            }
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (j0 + k < ed) {
                if ((unsigned)c[k] >= (unsigned)bn) {
                    bad = true;
                    c[k] = -1;
                } else {
                    ucfd::ld_values<B>(x + (int64_t)c[k]*B, xv[k]);
                }
            }
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (j0 + k < ed && c[k] >= 0) {
                double v = 0.0;
#pragma unroll
                for (int q = 0; q < B; ++q) v += a[k][q]*xv[k][q];
                arr += v;
            }
    }
    const int64_t o = (int64_t)i*B + r;
    y[o] = alpha*arr + beta*y[o];
    if (bad) ucfd::raise(flag, UCFD_KFLAG_INDEX);
}

__global__ __launch_bounds__(KB) void k_spmv_csr(int n, const int *__restrict__ rowptr,
                                                 const int *__restrict__ colidx,
                                                 const double *__restrict__ values, double alpha,
                                                 const double *__restrict__ x, double beta,
                                                 double *__restrict__ y, int *flag)
{
    const int i = kxcd()*KB + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    bool bad = false;
    for (int j = rowptr[i]; j < rowptr[i + 1]; ++j) {
        const int c = colidx[j];
        if ((unsigned)c < (unsigned)n) s += values[j]*x[c];
        else bad = true;
    }
    y[i] = alpha*s + beta*y[i];
    if (bad) ucfd::raise(flag, UCFD_KFLAG_INDEX);
}

template <int B>
__global__ __launch_bounds__(KB) void k_prepare(int bn, const int *__restrict__ diagslots,
                                                const double *__restrict__ values,
                                                double *__restrict__ dv, int *flag)
{
    const int i = blockIdx.x*KB + threadIdx.x;
    if (i >= bn) return;
    double a[B*B];
    const double *src = values + (int64_t)diagslots[i]*B*B;
#pragma unroll
    for (int q = 0; q < B*B; ++q) a[q] = src[q];
    if (!ucfd::ludcmp<B>(a)) ucfd::raise(flag, UCFD_KFLAG_PIVOT);
#pragma unroll
    for (int q = 0; q < B*B; ++q) dv[(int64_t)i*B*B + q] = a[q];
}

// ILU(0) factorisation, one level of rows per launch, one thread per row, in
// place on the values (ilu.c:4-48, bilu.c:5-65, pbilu.c:5-76 at one thread).
// For each lower slot k of row i, with ck = colidx[k]:
//   L_ik := A_ik U_kk^-1   (block: lusubmattrans with the factored diagonal
//                           block of row ck; scalar: division by its pivot)
//   A_ij -= L_ik A_{ck,j}  for each later slot j of row i whose column row ck
//                          also holds (the last such slot of row ck: the
//                          reference's marker array keeps the last write)
// then the block form factors its diagonal block in place (ludcmp).  dv gets
// the row's factored diagonal block (scalar: the pivot) for the solves.  A
// level holds rows that read only rows of earlier levels (complete) or of
// later ones (untouched), as the reference's row order has them.
template <int B, bool SCALAR>
__global__ __launch_bounds__(KB) void k_ilu_factor(int base, int cnt, const int *__restrict__ order,
                                                   const int *__restrict__ rowptr,
                                                   const int *__restrict__ colidx,
                                                   const int *__restrict__ diagslots,
                                                   double *values, double *__restrict__ dv,
                                                   int *flag)
{
    static_assert(!SCALAR || B == 1, "the scalar form has 1x1 blocks");
    constexpr int B2 = B*B;
    const int t = kxcd()*KB + threadIdx.x;
    if (t >= cnt) return;
    const int i = order ? order[base + t] : base + t;
    const int st = rowptr[i], ed = diagslots[i], jed = rowptr[i + 1];
    bool bad = false;
    for (int k = st; k < ed; ++k) {
        const int ck = colidx[k], kk = diagslots[ck], kst = rowptr[ck], ked = rowptr[ck + 1];
        double aik[B2];
        if (SCALAR) {
            const double p = values[kk];
            bad |= p == 0.0;
            aik[0] = values[k]/p;
            values[k] = aik[0];
        } else {
#pragma unroll
            for (int q = 0; q < B2; ++q) aik[q] = values[(int64_t)k*B2 + q];
            ucfd::lusubmattrans<B>(values + (int64_t)kk*B2, aik);
#pragma unroll
            for (int q = 0; q < B2; ++q) values[(int64_t)k*B2 + q] = aik[q];
        }
        for (int j = k + 1; j < jed; ++j) {
            const int col = colidx[j];
            int iwj = -1;
            for (int q = kst; q < ked; ++q)
                if (colidx[q] == col) iwj = q;
            if (iwj < 0) continue;
            if (SCALAR) {
                values[j] -= aik[0]*values[iwj];
                continue;
            }
            const double *u = values + (int64_t)iwj*B2;
            double *a = values + (int64_t)j*B2;
#pragma unroll
            for (int r = 0; r < B; ++r)
#pragma unroll
                for (int c = 0; c < B; ++c) {
                    double v = 0.0;
#pragma unroll
                    for (int e = 0; e < B; ++e) v += aik[r*B + e]*u[e*B + c];
                    a[r*B + c] -= v;
                }
        }
    }
    double d[B2];
#pragma unroll
    for (int q = 0; q < B2; ++q) d[q] = values[(int64_t)ed*B2 + q];
    if (SCALAR) {
        bad |= d[0] == 0.0;
    } else {
        bad |= !ucfd::ludcmp<B>(d);
#pragma unroll
        for (int q = 0; q < B2; ++q) values[(int64_t)ed*B2 + q] = d[q];
    }
#pragma unroll
    for (int q = 0; q < B2; ++q) dv[(int64_t)i*B2 + q] = d[q];
    if (bad) ucfd::raise(flag, UCFD_KFLAG_PIVOT);
}

// The block form on one wave per G = 64/B rows of a level: lane (g, r) owns
// scalar row r of block row g.  Both block operations of a lower slot act on
// rows independently: row r of L_ik = row r of A_ik times (L_kk U_kk)^-1
// (lusubmattrans restricted to one row, the same operations in the same
// order), and row r of A_ij -= (row r of L_ik) A_kj; so the lanes of a group
// run the row loop of the thread-per-row kernel side by side, reading the
// blocks of row ck whole (an earlier or a later level: not written here).
// The group then gathers its diagonal block with lane shuffles and every
// lane factors it; lane r writes row r.  Bit-identical to k_ilu_factor.
// Requires that no lower slot of a row refers to the row itself (the host
// keeps k_ilu_factor for such a matrix).
// Bound by the chain over the lower slots.  The search for a slot's column in the
// pivot row was a load per entry and slot; the columns are now in LDS before the
// chain starts (rows beyond IS entries take the rest from memory) and the blocks are
// read in wide loads: a level of 2.1K rows with six lower slots 40.7 -> 21.7 us.
template <int B>
__global__ __launch_bounds__(64) void k_ilu_factor_w(int base, int cnt,
                                                     const int *__restrict__ order,
                                                     const int *__restrict__ rowptr,
                                                     const int *__restrict__ colidx,
                                                     const int *__restrict__ diagslots,
                                                     double *values, double *__restrict__ dv,
                                                     int *flag)
{
    constexpr int B2 = B*B, G = 64/B;
    constexpr int IS = 8;   // entries of a row whose columns are held
    __shared__ int scol[G + 1][IS], sdiag[G + 1][IS], sst[G + 1][IS], sed[G + 1][IS];
    __shared__ int sk[G + 1][IS][IS];
    const int lane = threadIdx.x;
    const int t0 = ucfd::wave_xcd_index()*G;
    if (t0 >= cnt) return;
    const int g = lane/B, r = lane%B;
    const bool act = g < G && t0 + g < cnt;
    int i = 0, st = 0, ed = 0, jed = 0;
    if (act) {
        i = order ? order[base + t0 + g] : base + t0 + g;
        st = rowptr[i];
        ed = diagslots[i];
        jed = rowptr[i + 1];
    }
    // the columns of the row's first IS entries and, for each of its lower slots
    // among them, the diagonal slot and the first IS columns of the slot's row: three
    // round trips for all of them, met by the lanes of the group side by side
    const int nrow = min(jed - st, IS), nlow = min(ed - st, IS);
    if (act)
        for (int q = r; q < nrow; q += B) scol[g][q] = colidx[st + q];
    ucfd::wave_lds_sync();
    if (act)
        for (int q = r; q < nlow; q += B) {
            const int c = scol[g][q];
            sdiag[g][q] = diagslots[c];
            sst[g][q] = rowptr[c];
            sed[g][q] = rowptr[c + 1];
        }
    ucfd::wave_lds_sync();
    if (act)
        for (int q = r; q < nlow*IS; q += B) {
            const int j = sst[g][q/IS] + q%IS;
            sk[g][q/IS][q%IS] = j < sed[g][q/IS] ? colidx[j] : -1;
        }
    ucfd::wave_lds_sync();
    for (int k = st; k < ed; ++k) {
        const int p = k - st;
        const bool held = p < IS;
        int kk, kst, ked, kcol[IS];
        if (held) {
            kk = sdiag[g][p];
            kst = sst[g][p];
            ked = sed[g][p];
#pragma unroll
            for (int q = 0; q < IS; ++q) kcol[q] = sk[g][p][q];
        } else {
            const int ck = colidx[k];
            kk = diagslots[ck];
            kst = rowptr[ck];
            ked = rowptr[ck + 1];
#pragma unroll
            for (int q = 0; q < IS; ++q) kcol[q] = kst + q < ked ? colidx[kst + q] : -1;
        }
        double m[B], LU[B2];
        ucfd::ld_values<B>(values + (int64_t)k*B2 + r*B, m);
        ucfd::ld_values<B2>(values + (int64_t)kk*B2, LU);
        // row r of M (L U)^-1, in the order of ucfd::lusubmattrans
        m[0] /= LU[0];
#pragma unroll
        for (int c = 1; c < B; ++c) {
            double val = 0.0;
#pragma unroll
            for (int q = 0; q < c; ++q) val += m[q]*LU[q*B + c];
            m[c] = (m[c] - val)/LU[c*B + c];
        }
#pragma unroll
        for (int c = B - 2; c > -1; --c) {
            double val = 0.0;
#pragma unroll
            for (int q = c + 1; q < B; ++q) val += m[q]*LU[q*B + c];
            m[c] -= val;
        }
#pragma unroll
        for (int c = 0; c < B; ++c) values[(int64_t)k*B2 + r*B + c] = m[c];
        for (int j = k + 1; j < jed; ++j) {
            const int col = j - st < IS ? scol[g][j - st] : colidx[j];
            int iwj = -1;
#pragma unroll
            for (int q = 0; q < IS; ++q)
                if (kcol[q] == col) iwj = kst + q;
            for (int q = kst + IS; q < ked; ++q)
                if (colidx[q] == col) iwj = q;
            if (iwj < 0) continue;
            double u[B2], a[B];
            ucfd::ld_values<B2>(values + (int64_t)iwj*B2, u);
            ucfd::ld_values<B>(values + (int64_t)j*B2 + r*B, a);
#pragma unroll
            for (int c = 0; c < B; ++c) {
                double v = 0.0;
#pragma unroll
                for (int e = 0; e < B; ++e) v += m[e]*u[e*B + c];
                values[(int64_t)j*B2 + r*B + c] = a[c] - v;
            }
        }
    }
    // the group's diagonal block (each lane wrote its own row), then LU
    double dr[B];
#pragma unroll
    for (int c = 0; c < B; ++c) dr[c] = act ? values[(int64_t)ed*B2 + r*B + c] : 0.0;
    double d[B2];
#pragma unroll
    for (int rr = 0; rr < B; ++rr)
#pragma unroll
        for (int c = 0; c < B; ++c) d[rr*B + c] = __shfl(dr[c], g*B + rr, 64);
    if (!act) return;
    if (!ucfd::ludcmp<B>(d) && r == 0) ucfd::raise(flag, UCFD_KFLAG_PIVOT);
    double o[B];
#pragma unroll
    for (int c = 0; c < B; ++c) o[c] = d[c];
#pragma unroll
    for (int rr = 1; rr < B; ++rr)
        if (r == rr)
#pragma unroll
            for (int c = 0; c < B; ++c) o[c] = d[rr*B + c];
#pragma unroll
    for (int c = 0; c < B; ++c) {
        values[(int64_t)ed*B2 + r*B + c] = o[c];
        dv[(int64_t)i*B2 + r*B + c] = o[c];
    }
}

__global__ void k_to32(int64_t n, const double *__restrict__ a, float *__restrict__ b)
{
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t j = (int64_t)blockIdx.x*KB + threadIdx.x; j < n; j += st) b[j] = (float)a[j];
}

// ----------------------------------------------------------- block sweeps
//
// Sweep kinds (template parameter K) of the FP64 kernels:
//   SW_LUSGS  block LU-SGS (blusgs.c:28-100): lower x_i = D_i^-1 (b_i -
//             sum_{j<diag} A_ij x_j); upper x_i -= D_i^-1 sum_{j>diag} A_ij x_j
//   SW_BILU   block ILU(0) solve with the factored blocks (bilu.c:67-130):
//             lower x_i = b_i - sum_{j<diag} L_ij x_j; upper x_i = U_ii^-1
//             (x_i - sum_{j>diag} U_ij x_j), U_ii^-1 by LU substitution
//   SW_ILU    scalar ILU(0) solve (ilu.c:50-86, B = 1): the same with the
//             products subtracted one by one and a division by U_ii
constexpr int SW_LUSGS = KRY_SW_LUSGS, SW_BILU = KRY_SW_BILU, SW_ILU = KRY_SW_ILU;

template <int B, bool UPPER, int K>
__global__ __launch_bounds__(KB) void k_sweep64(int base, int cnt, const int *__restrict__ order,
                                                const int *__restrict__ rowptr,
                                                const int *__restrict__ colidx,
                                                const int *__restrict__ diagslots,
                                                const double *__restrict__ values,
                                                const double *__restrict__ dv, double *b)
{
    static_assert(K != SW_ILU || B == 1, "the scalar ILU solve has 1x1 blocks");
    const int t = kxcd()*KB + threadIdx.x;
    if (t >= cnt) return;
    const int i = order ? order[base + t] : base + t;
    const int dd = diagslots[i];
    double arr[B];
    if (!UPPER || K != SW_LUSGS) {
#pragma unroll
        for (int k = 0; k < B; ++k) arr[k] = b[(int64_t)i*B + k];
    } else {
#pragma unroll
        for (int k = 0; k < B; ++k) arr[k] = 0.0;
    }
    const int j0 = UPPER ? dd + 1 : rowptr[i];
    const int j1 = UPPER ? rowptr[i + 1] : dd;
    for (int j = j0; j < j1; ++j) {
        const int c = colidx[j];
        if (K == SW_ILU) {
            arr[0] -= __builtin_nontemporal_load(values + j)*b[c];
            continue;
        }
        const double *blk = values + (int64_t)j*B*B;
        double xc[B];
#pragma unroll
        for (int q = 0; q < B; ++q) xc[q] = b[(int64_t)c*B + q];
#pragma unroll
        for (int r = 0; r < B; ++r) {
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < B; ++q) v += __builtin_nontemporal_load(blk + r*B + q)*xc[q];
            if (UPPER && K == SW_LUSGS) arr[r] += v;
            else arr[r] -= v;
        }
    }
    if (K != SW_LUSGS && !UPPER) {
#pragma unroll
        for (int k = 0; k < B; ++k) b[(int64_t)i*B + k] = arr[k];
        return;
    }
    if (K == SW_ILU) {
        b[i] = arr[0]/dv[i];
        return;
    }
    double lu[B*B];
#pragma unroll
    for (int q = 0; q < B*B; ++q) lu[q] = __builtin_nontemporal_load(dv + (int64_t)i*B*B + q);
    ucfd::lusub<B>(lu, arr);
#pragma unroll
    for (int k = 0; k < B; ++k) {
        const int64_t o = (int64_t)i*B + k;
        if (UPPER && K == SW_LUSGS) b[o] -= arr[k];
        else b[o] = arr[k];
    }
}

template <int B, bool UPPER>
__global__ __launch_bounds__(KB) void k_sweep32(int base, int cnt, const int *__restrict__ order,
                                                const int *__restrict__ rowptr,
                                                const int *__restrict__ colidx,
                                                const int *__restrict__ diagslots,
                                                const float *__restrict__ v32,
                                                const double *__restrict__ dv, float *x32,
                                                double *b)
{
    const int t = kxcd()*KB + threadIdx.x;
    if (t >= cnt) return;
    const int i = order ? order[base + t] : base + t;
    const int dd = diagslots[i];
    float acc[B];
#pragma unroll
    for (int k = 0; k < B; ++k) acc[k] = 0.0f;
    const int j0 = UPPER ? dd + 1 : rowptr[i];
    const int j1 = UPPER ? rowptr[i + 1] : dd;
    for (int j = j0; j < j1; ++j) {
        const int c = colidx[j];
        const float *blk = v32 + (int64_t)j*B*B;
        float xc[B];
#pragma unroll
        for (int q = 0; q < B; ++q) xc[q] = x32[(int64_t)c*B + q];
#pragma unroll
        for (int r = 0; r < B; ++r) {
            float v = 0.0f;
#pragma unroll
            for (int q = 0; q < B; ++q) v += __builtin_nontemporal_load(blk + r*B + q)*xc[q];
            acc[r] += v;
        }
    }
    double lu[B*B], arr[B];
#pragma unroll
    for (int q = 0; q < B*B; ++q) lu[q] = __builtin_nontemporal_load(dv + (int64_t)i*B*B + q);
    if (!UPPER) {
#pragma unroll
        for (int k = 0; k < B; ++k) arr[k] = b[(int64_t)i*B + k] - (double)acc[k];
        ucfd::lusub<B>(lu, arr);
#pragma unroll
        for (int k = 0; k < B; ++k) x32[(int64_t)i*B + k] = (float)arr[k];
    } else {
#pragma unroll
        for (int k = 0; k < B; ++k) arr[k] = (double)acc[k];
        ucfd::lusub<B>(lu, arr);
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const int64_t o = (int64_t)i*B + k;
            const double v = (double)x32[o] - arr[k];
            x32[o] = (float)v;
            b[o] = v;
        }
    }
}

// Block sweeps on one wave per G = 64/B rows of a contiguous row range
// (block sizes 2..7).  Lane (g, r) accumulates scalar row r of row g over
// the row's lower (lower sweep) or upper (upper sweep) blocks in the order
// of k_sweep64 / k_sweep32 above; the group then exchanges its B sums with
// lane shuffles and every lane runs the row's diagonal solve (bit-identical
// to the thread-per-row kernels).  K selects the FP64 sweep kind (SW_LUSGS
// or SW_BILU; the mixed form is LU-SGS only).  Blocks, neighbour rows and the LU
// block are read in the widest loads that cover them, the LU block with the
// row's first indices (it depends on nothing else) and KP blocks together, so a
// row of up to KP blocks is three round trips: indices, blocks and column
// indices, neighbour rows.  One apply (FP32 products / FP64 / block ILU), blocks
// staged through LDS -> this: 4.9K hex rows 22/21/18 -> 14/14/13 us, 64K
// 40.6/35.0/29.3 -> 24.5/29.7/24.8, 384K tet rows, 4 colours, 117/150/133 ->
// 105/129/111, 1M, 2 colours, 222/305/265 -> 208/286/238; 7x7 blocks, 384K rows,
// 186/243/201 -> 154/215/171.
//
// The LU block: from 5x5 on each lane reads its own row and the group exchanges
// the rows by shuffles after the sums (every lane holding the whole block from
// the start: 384K rows 106/135/115 -> 105/129/111 us, 1M 220/300/244 ->
// 208/286/238, 7x7 173/228/178 -> 154/215/171); smaller blocks are read whole
// (4x4: 51/67/57 against 53/66/57).
template <int B> constexpr bool lu_rows() { return B >= 5; }

template <int B> __device__ __forceinline__ void ld_lu(const double *p, int r, double *lu)
{
    if (lu_rows<B>()) ucfd::ld_values<B>(p + r*B, lu);   // lu[0 .. B-1]: row r
    else ucfd::ld_values<B*B>(p, lu);
}

// the whole block in every lane of group g (all lanes of the wave take part)
template <int B> __device__ __forceinline__ void share_lu(int g, double *lu)
{
    if (!lu_rows<B>()) return;
    double row[B];
#pragma unroll
    for (int c = 0; c < B; ++c) row[c] = lu[c];
#pragma unroll
    for (int rr = 0; rr < B; ++rr)
#pragma unroll
        for (int c = 0; c < B; ++c) lu[rr*B + c] = __shfl(row[c], g*B + rr, 64);
}

// JOIN (a lower sweep): the row's update of the upper sweep follows, for rows with
// no block above the diagonal (k_bsgs_diag's expressions on the values just formed,
// so the same bits).  It saves the launch of 2.8 us for
// 2.1K rows (ILU, 8 of them a solve), 4.2 us of 31K rows (LU-SGS in FP32).
template <int B, bool UPPER, bool F32, int K, bool JOIN = false>
__global__ __launch_bounds__(64) void k_bsgs_w(int base, int cnt, const int *__restrict__ rowptr,
                                               const int *__restrict__ colidx,
                                               const int *__restrict__ diagslots,
                                               const typename std::conditional<F32, float,
                                                                               double>::type
                                                   *__restrict__ vals,
                                               const double *__restrict__ dv, float *x32,
                                               double *b)
{
    using T = typename std::conditional<F32, float, double>::type;
    static_assert(K == SW_LUSGS || (K == SW_BILU && !F32), "sweep kind");
    constexpr int B2 = B*B, G = 64/B, KP = 4;
    // LU-SGS adds the upper products and applies D^-1 to the sum, the others
    // subtract from x_i; the lower ILU sweep has no diagonal solve
    constexpr bool ADD = UPPER && K == SW_LUSGS, SOLVE = K != SW_BILU || UPPER;
    static_assert(!JOIN || !UPPER, "a lower sweep joins the upper one");
    const int lane = threadIdx.x;
    const int t0 = ucfd::wave_xcd_index()*G;
    if (t0 >= cnt) return;
    const int g = lane/B, r = lane%B;
    const int i = base + t0 + g;
    const bool act = g < G && t0 + g < cnt;
    const int64_t o = (int64_t)i*B + r;
    int j0 = 0, j1 = 0;
    double lu[B2] = {}, own = 0.0;
    float own32 = 0.0f;
    if (act) {
        const int dd = diagslots[i];
        j0 = UPPER ? dd + 1 : rowptr[i];
        j1 = UPPER ? rowptr[i + 1] : dd;
        if (SOLVE || JOIN) ld_lu<B>(dv + (int64_t)i*B2, r, lu);
        if (F32 && UPPER) own32 = x32[o];
        else own = b[o];
    }
    T acc = T(0);
    double a = !F32 && !ADD ? own : 0.0;
    for (int jj = j0; jj < j1; jj += KP) {
        int c[KP];
        T blk[KP][B], xc[KP][B];
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (jj + k < j1) {
                c[k] = colidx[jj + k];
                ucfd::ld_values<B>(vals + (int64_t)(jj + k)*B2 + r*B, blk[k]);
            }
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (jj + k < j1) {
                if constexpr (F32) ucfd::ld_values<B>(x32 + (int64_t)c[k]*B, xc[k]);
                else ucfd::ld_values<B>(b + (int64_t)c[k]*B, xc[k]);
            }
#pragma unroll
        for (int k = 0; k < KP; ++k)
            if (jj + k < j1) {
                T v = T(0);
#pragma unroll
                for (int q = 0; q < B; ++q) v += blk[k][q]*xc[k][q];
                if (F32) acc += v;
                else if (ADD) a += (double)v;
                else a -= (double)v;
            }
    }
    if (!SOLVE && !JOIN) {
        if (act) b[o] = a;
        return;
    }
    if (F32) {
        if (UPPER) a = (double)acc;
        else if (act) a = own - (double)acc;
    }
    // the group's B sums, then the diagonal solve in every lane of the group
    double arr[B];
#pragma unroll
    for (int k = 0; k < B; ++k) arr[k] = __shfl(a, g*B + k, 64);
    share_lu<B>(g, lu);
    if (!act) return;
    ucfd::lusub<B>(lu, arr);
    double mine = arr[0];
#pragma unroll
    for (int k = 1; k < B; ++k)
        if (r == k) mine = arr[k];
    if (JOIN && K == SW_LUSGS) {
        // the upper update with an empty sum
        if (F32) own32 = (float)mine;
        else own = mine;
        const double zero = F32 ? (double)0.0f : 0.0;
#pragma unroll
        for (int k = 0; k < B; ++k) arr[k] = zero;
        ucfd::lusub<B>(lu, arr);
        mine = arr[0];
#pragma unroll
        for (int k = 1; k < B; ++k)
            if (r == k) mine = arr[k];
    }
    if (F32) {
        if (UPPER || JOIN) {
            const double v = (double)own32 - mine;
            x32[o] = (float)v;
            b[o] = v;
        } else {
            x32[o] = (float)mine;
        }
    } else {
        b[o] = ADD || (JOIN && K == SW_LUSGS) ? own - mine : mine;
    }
}

// A level whose rows take no block in the sweep's direction (the first
// colour of a lower sweep, the last of an upper one): k_bsgs_w's row update
// with an empty product sum, its expressions kept literally (a = b - 0 for
// the FP32 lower sweep, a = 0 for the LU-SGS upper one), so the bits are
// the same.  The row's own entries and its LU block are requested together
// at the start, with no index loads in front of them: one memory round trip
// per wave instead of three.  (The lower BILU sweep of such a level leaves
// b unchanged and is not launched.)
template <int B, bool UPPER, bool F32, int K>
__global__ __launch_bounds__(64) void k_bsgs_diag(int base, int cnt, const double *__restrict__ dv,
                                                  float *x32, double *b)
{
    constexpr int B2 = B*B, G = 64/B;
    constexpr bool ADD = UPPER && K == SW_LUSGS;
    static_assert(K == SW_LUSGS || (K == SW_BILU && UPPER && !F32), "sweep kind");
    const int lane = threadIdx.x;
    const int t0 = ucfd::wave_xcd_index()*G;
    if (t0 >= cnt) return;
    const int g = lane/B, r = lane%B;
    const int i = base + t0 + g;
    const bool act = g < G && t0 + g < cnt;
    const int64_t o = (int64_t)i*B + r;
    double lu[B2] = {}, bo = 0.0;
    float xo = 0.f;
    if (act) {
        ld_lu<B>(dv + (int64_t)i*B2, r, lu);
        if (!ADD) bo = b[o];
        if (F32 && UPPER) xo = x32[o];
    }
    double a = 0.0;
    if (!F32 && !ADD && act) a = bo;
    if (F32) {
        if (UPPER) a = (double)0.0f;
        else if (act) a = bo - (double)0.0f;
    }
    double arr[B];
#pragma unroll
    for (int k = 0; k < B; ++k) arr[k] = __shfl(a, g*B + k, 64);
    share_lu<B>(g, lu);
    if (!act) return;
    ucfd::lusub<B>(lu, arr);
    double mine = arr[0];
#pragma unroll
    for (int k = 1; k < B; ++k)
        if (r == k) mine = arr[k];
    if (F32) {
        if (UPPER) {
            const double v = (double)xo - mine;
            x32[o] = (float)v;
            b[o] = v;
        } else {
            x32[o] = (float)mine;
        }
    } else {
        if (ADD) b[o] = b[o] - mine;
        else b[o] = mine;
    }
}

// --------------------------------------------------------------- BLAS
__device__ __forceinline__ double block_reduce(double v)
{
    __shared__ double red[KB/64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (threadIdx.x % 64 == 0) red[threadIdx.x/64] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < KB/64; ++w) s += red[w];
    __syncthreads();
    return s;
}

// Sum of row part[0 .. np-1] (np <= KMAXPART) by one wave, in every lane: the
// sums of 64 consecutive partials (a fixed tree), added in order.
__device__ __forceinline__ double wave_row_sum(const double *__restrict__ part, int np)
{
    constexpr int U = 8;
    const int lane = threadIdx.x & 63;
    double t = 0.0;
    for (int q0 = 0; q0 < np; q0 += 64*U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = q0 + u*64 + lane;
            v[u] = j < np ? part[j] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (q0 + u*64 >= np) break;
            for (int o = 32; o > 0; o >>= 1) v[u] += __shfl_xor(v[u], o, 64);
            t += v[u];
        }
    }
    return t;
}

// hs[j] = the sum of row j of the partials, j < k, by the workgroup.  A kernel
// that needs the result of a reduction sums its partials itself, every
// workgroup for itself, when there are at most KFUSE a row: 21K unknowns, 83
// partials a row, save a launch and its gap (2.3 + 1.5 us) for under 1 us.  With
// 1024 a row the sums cost 8 us (k = 4) to 17 us (k = 10) where the launch costs
// 4.7, so longer rows are summed to one value by k_sum_rows first.
constexpr int KFUSE = 256;

__device__ __forceinline__ void block_row_sums(double *hs, const double *__restrict__ part, int np,
                                               int k)
{
    for (int j = threadIdx.x >> 6; j < k; j += KB/64) {
        const double t = wave_row_sum(part + (int64_t)j*KMAXPART, np);
        if ((threadIdx.x & 63) == 0) hs[j] = t;
    }
    __syncthreads();
}

// Scalars for the host: written to pinned memory by the first workgroup, the
// sequence number last (KryPost::seq 0: more values follow from a later kernel)
__device__ __forceinline__ void post(const KryPost &h, const double *v, int k)
{
    if (blockIdx.x != 0 || threadIdx.x != 0 || !h.out) return;
    for (int j = 0; j < k; ++j)
        __hip_atomic_store(h.out + j, v[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (h.seq)
        __hip_atomic_store(h.word, h.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// one workgroup per row: the row's sum replaces its first partial
__global__ __launch_bounds__(1024) void k_sum_rows(double *part, int np)
{
    __shared__ double red[16];
    double *p = part + (int64_t)blockIdx.x*KMAXPART;
    double s = (int)threadIdx.x < np ? p[threadIdx.x] : 0.0;
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (threadIdx.x % 64 == 0) red[threadIdx.x/64] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < 16; ++w) t += red[w];
        p[0] = t;
    }
}

// one row's sum, to out (device) and to the host
__global__ __launch_bounds__(64) void k_sum_row(const double *part, int np, double *out, KryPost h)
{
    const double t = wave_row_sum(part, np);
    if (threadIdx.x == 0) *out = t;
    post(h, &t, 1);
}

__global__ __launch_bounds__(KB) void k_dot(int64_t n, const double *__restrict__ x,
                                            const double *__restrict__ y, double *part)
{
    double s = 0.0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) s += x[i]*y[i];
    s = block_reduce(s);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(KB) void k_dot5(int64_t n, const double *__restrict__ rt,
                                             const double *__restrict__ sv,
                                             const double *__restrict__ t, double *part)
{
    double a = 0, b = 0, c = 0, d = 0, e = 0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        const double sk = sv[i], tk = t[i], rk = rt[i];
        a += rk*sk; b += rk*tk; c += tk*sk; d += tk*tk; e += sk*sk;
    }
    const double v[5] = {a, b, c, d, e};
    for (int q = 0; q < 5; ++q) {
        const double r = block_reduce(v[q]);
        if (threadIdx.x == 0) part[q*KMAXPART + blockIdx.x] = r;
    }
}

// partial dots of w with V columns j0..j0+7 (fewer at the end)
__global__ __launch_bounds__(KB) void k_gemvt8(int64_t n, int k, int j0, const double *__restrict__ V,
                                               int64_t ldv, const double *__restrict__ w,
                                               double *part)
{
    double acc[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] = 0.0;
    const int nj = k - j0 < 8 ? k - j0 : 8;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        const double wi = w[i];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (q < nj) acc[q] += V[(int64_t)(j0 + q)*ldv + i]*wi;
    }
    for (int q = 0; q < nj; ++q) {
        const double r = block_reduce(acc[q]);
        if (threadIdx.x == 0) part[(int64_t)(j0 + q)*KMAXPART + blockIdx.x] = r;
    }
}

// w += alpha V h, h the sums of the partials hpart (posted to the host), and
// with part the partials of |w|^2.  Any k <= 64.
__global__ __launch_bounds__(KB) void k_gemv(int64_t n, int k, const double *__restrict__ V,
                                             int64_t ldv, double alpha,
                                             const double *__restrict__ hpart, int np,
                                             double *__restrict__ w, double *part, KryPost post_h)
{
    __shared__ double hs[64];
    block_row_sums(hs, hpart, np, k);
    post(post_h, hs, k);
    double ss = 0.0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double sum = 0.0;
        for (int j = 0; j < k; ++j) sum += V[(int64_t)j*ldv + i]*hs[j];
        const double v = alpha*sum + 1.0*w[i];
        w[i] = v;
        ss += v*v;
    }
    if (part) {
        ss = block_reduce(ss);
        if (threadIdx.x == 0) part[blockIdx.x] = ss;
    }
}

// k_gemv for k <= KM columns with the row of V loaded into registers first
// (every load issued before the first product; the same sums in the same
// order)
template <int KM>
__global__ __launch_bounds__(KB) void k_gemv_r(int64_t n, int k, const double *__restrict__ V,
                                               int64_t ldv, double alpha,
                                               const double *__restrict__ hpart, int np,
                                               double *__restrict__ w, double *part,
                                               KryPost post_h)
{
    __shared__ double hs[KM];
    block_row_sums(hs, hpart, np, k);
    post(post_h, hs, k);
    double ss = 0.0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double vr[KM];
#pragma unroll
        for (int q = 0; q < KM; ++q) vr[q] = q < k ? V[(int64_t)q*ldv + i] : 0.0;
        double sum = 0.0;
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) sum += vr[q]*hs[q];
        const double v = alpha*sum + 1.0*w[i];
        w[i] = v;
        ss += v*v;
    }
    if (part) {
        ss = block_reduce(ss);
        if (threadIdx.x == 0) part[blockIdx.x] = ss;
    }
}

// x += V y with the coefficients in the launch's arguments (no copy to the
// device): k_gemv's sums, KM columns at a time with their loads issued together
template <int KM>
__global__ __launch_bounds__(KB) void k_gemv_y(int64_t n, int k, const double *__restrict__ V,
                                               int64_t ldv, KryCoef y, double *__restrict__ x)
{
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double sum = 0.0;
        for (int j = 0; j < k; j += KM) {
            double vr[KM];
#pragma unroll
            for (int q = 0; q < KM; ++q) vr[q] = j + q < k ? V[(int64_t)(j + q)*ldv + i] : 0.0;
#pragma unroll
            for (int q = 0; q < KM; ++q)
                if (j + q < k) sum += vr[q]*y.v[j + q];
        }
        x[i] = 1.0*sum + 1.0*x[i];
    }
}

// partial dots of w with all k <= KM columns of V in one pass over w (each
// column's sum runs over the same elements in the same order as k_gemvt8's)
template <int KM>
__global__ __launch_bounds__(KB) void k_gemvt_all(int64_t n, int k, const double *__restrict__ V,
                                                  int64_t ldv, const double *__restrict__ w,
                                                  double *part)
{
    double acc[KM];
#pragma unroll
    for (int q = 0; q < KM; ++q) acc[q] = 0.0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        // the row of V first, every load issued before the first product
        double vr[KM];
#pragma unroll
        for (int q = 0; q < KM; ++q) vr[q] = q < k ? V[(int64_t)q*ldv + i] : 0.0;
        const double wi = w[i];
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) acc[q] += vr[q]*wi;
    }
#pragma unroll
    for (int q = 0; q < KM; ++q)
        if (q < k) {
            const double r = block_reduce(acc[q]);
            if (threadIdx.x == 0) part[(int64_t)q*KMAXPART + blockIdx.x] = r;
        }
}

// The middle of a CGS2 step in one pass over V: w_i += alpha*sum_j V_ji h_j
// (k_gemv's arithmetic), then partial dots of the new w with the same k <= KM
// columns (k_gemvt_all's), the row of V held in registers between the two.
template <int KM>
__global__ __launch_bounds__(KB) void k_gemv_gemvt(int64_t n, int k,
                                                   const double *__restrict__ V, int64_t ldv,
                                                   double alpha,
                                                   const double *__restrict__ hpart, int np,
                                                   double *__restrict__ w, double *part,
                                                   KryPost post_h)
{
    __shared__ double hs[KM];
    block_row_sums(hs, hpart, np, k);
    post(post_h, hs, k);
    double acc[KM];
#pragma unroll
    for (int q = 0; q < KM; ++q) acc[q] = 0.0;
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double vr[KM];
#pragma unroll
        for (int q = 0; q < KM; ++q) vr[q] = q < k ? V[(int64_t)q*ldv + i] : 0.0;
        double sum = 0.0;
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) sum += vr[q]*hs[q];
        const double v = alpha*sum + 1.0*w[i];
        w[i] = v;
#pragma unroll
        for (int q = 0; q < KM; ++q)
            if (q < k) acc[q] += vr[q]*v;
    }
#pragma unroll
    for (int q = 0; q < KM; ++q)
        if (q < k) {
            const double r = block_reduce(acc[q]);
            if (threadIdx.x == 0) part[(int64_t)q*KMAXPART + blockIdx.x] = r;
        }
}

// dst = src/sqrt(sum of the partials nsq), the sum posted to the host
__global__ __launch_bounds__(KB) void k_scale_isqrt(int64_t n, const double *__restrict__ src,
                                                    const double *__restrict__ nsq, int np,
                                                    double *__restrict__ dst,
                                                    double *__restrict__ dst2, KryPost post_n)
{
    __shared__ double hs[1];
    block_row_sums(hs, nsq, np, 1);
    post(post_n, hs, 1);
    const double inv = 1.0/sqrt(hs[0]);
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        const double v = inv*src[i];
        dst[i] = v;
        if (dst2) dst2[i] = v;
    }
}

__global__ __launch_bounds__(KB) void k_axpby(int64_t n, double a, const double *__restrict__ x,
                                              double b, double *__restrict__ y, int mode)
{
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        if (mode == 0) y[i] += a*x[i];          // axpy
        else if (mode == 1) y[i] = a*x[i] + b*y[i];
        else if (mode == 2) y[i] = x[i];        // copy
        else y[i] = a;                          // fill
    }
}

__global__ __launch_bounds__(KB) void k_bicg_p(int64_t n, double beta, double omega,
                                               const double *__restrict__ r,
                                               const double *__restrict__ v,
                                               double *__restrict__ p, double *__restrict__ pt)
{
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double t = p[i] + (-omega)*v[i];
        t = beta*t;
        t = t + 1.0*r[i];
        p[i] = t;
        pt[i] = t;
    }
}

// s = r - alpha*v (as copy + axpy); shat = s
// alpha = rho/pi with pi the sum of the partials (the host forms the same
// quotient once it has pi)
__global__ __launch_bounds__(KB) void k_bicg_s(int64_t n, double rho,
                                               const double *__restrict__ pi_part, int np,
                                               const double *__restrict__ r,
                                               const double *__restrict__ v,
                                               double *__restrict__ sv, double *__restrict__ shat)
{
    __shared__ double hs[1];
    block_row_sums(hs, pi_part, np, 1);
    const double alpha = rho/hs[0];
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        const double t = r[i] + (-alpha)*v[i];
        sv[i] = t;
        shat[i] = t;
    }
}

__global__ __launch_bounds__(KB) void k_cast32(int64_t n, const double *__restrict__ a,
                                               float *__restrict__ b)
{
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) b[i] = (float)a[i];
}

// The end of a BiCGSTAB iteration: pi and the five dots summed from their
// partials and posted to the host, alpha = rho/pi and omega = (t.s)/(t.t) formed
// here as the host forms them, then x += alpha pt + omega shat, r = s - omega t.
// A pi breakdown (bicgstab.c:84) leaves x and r as they are.
__global__ __launch_bounds__(KB) void k_bicg_xr(int64_t n, double rho,
                                                const double *__restrict__ pi_part,
                                                const double *__restrict__ dots, int np,
                                                const double *__restrict__ pt,
                                                const double *__restrict__ shat,
                                                const double *__restrict__ sv,
                                                const double *__restrict__ t,
                                                double *__restrict__ x, double *__restrict__ r,
                                                KryPost post_d)
{
    __shared__ double hs[6];
    block_row_sums(hs, dots, np, 5);
    block_row_sums(hs + 5, pi_part, np, 1);
    post(post_d, hs, 6);
    const double pi = hs[5];
    if (fabs(pi) < 1e-30) return;
    const double alpha = rho/pi, omega = hs[2]/hs[3];
    const int64_t st = (int64_t)gridDim.x*KB;
    for (int64_t i = (int64_t)blockIdx.x*KB + threadIdx.x; i < n; i += st) {
        double xv = x[i] + alpha*pt[i];
        x[i] = xv + omega*shat[i];
        r[i] = sv[i] + (-omega)*t[i];
    }
}

int ok() { return hipGetLastError() == hipSuccess ? UCFD_OK : UCFD_ERR_HIP; }

template <template <int> class F, typename... A>
int by_block(int blk, A... a)
{
    switch (blk) {
    case 1: return F<1>::run(a...);
    case 2: return F<2>::run(a...);
    case 3: return F<3>::run(a...);
    case 4: return F<4>::run(a...);
    case 5: return F<5>::run(a...);
    case 6: return F<6>::run(a...);
    case 7: return F<7>::run(a...);
    default: return UCFD_ERR_ARG;
    }
}

template <int B> struct SpmvL {
    static int run(hipStream_t s, int bn, const int *rp, const int *ci, const double *v, double al,
                   const double *x, double be, double *y, int *flag)
    {
        if (B == 1) {
            hipLaunchKernelGGL(k_spmv_bsr<B>, dim3((bn + KB - 1)/KB), dim3(KB), 0, s, bn, rp, ci,
                               v, al, x, be, y, flag);
        } else {
            constexpr int G = 64/B;
            hipLaunchKernelGGL(k_spmv_bsr_w<B>, dim3((bn + G - 1)/G), dim3(64), 0, s, bn, rp, ci,
                               v, al, x, be, y, flag);
        }
        return ok();
    }
};

template <int B> struct PrepL {
    static int run(hipStream_t s, int bn, const int *ds, const double *v, double *dv, int *flag)
    {
        hipLaunchKernelGGL(k_prepare<B>, dim3((bn + KB - 1)/KB), dim3(KB), 0, s, bn, ds, v, dv,
                           flag);
        return ok();
    }
};

template <int B> struct IluL {
    static int run(hipStream_t s, bool scalar, bool rows, int base, int cnt, const int *ord,
                   const int *rp, const int *ci, const int *ds, double *v, double *dv, int *flag)
    {
        const dim3 g((cnt + KB - 1)/KB);
        if (scalar) {
            if (B != 1) return UCFD_ERR_ARG;
            hipLaunchKernelGGL((k_ilu_factor<1, true>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci,
                               ds, v, dv, flag);
        } else if (B > 1 && rows) {
            if constexpr (B > 1)
                hipLaunchKernelGGL((k_ilu_factor_w<B>), dim3((cnt + 64/B - 1)/(64/B)), dim3(64), 0,
                                   s, base, cnt, ord, rp, ci, ds, v, dv, flag);
        } else {
            hipLaunchKernelGGL((k_ilu_factor<B, false>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci,
                               ds, v, dv, flag);
        }
        return ok();
    }
};

template <int B, int K>
int sweep64_launch(hipStream_t s, int upper, int base, int cnt, const int *ord, const int *rp,
                   const int *ci, const int *ds, const double *v, const double *dv, double *b,
                   bool empty, bool join)
{
    if constexpr (B > 1) {
        if (!ord) {
            const dim3 g((cnt + 64/B - 1)/(64/B));
            if (empty && K != SW_ILU) {
                // no row of the level takes a block in this direction
                if (K == SW_BILU && !upper) return UCFD_OK;
                if (upper)
                    hipLaunchKernelGGL((k_bsgs_diag<B, true, false, K>), g, dim3(64), 0, s, base,
                                       cnt, dv, nullptr, b);
                else if constexpr (K == SW_LUSGS)
                    hipLaunchKernelGGL((k_bsgs_diag<B, false, false, K>), g, dim3(64), 0, s, base,
                                       cnt, dv, nullptr, b);
                return ok();
            }
            if (upper)
                hipLaunchKernelGGL((k_bsgs_w<B, true, false, K>), g, dim3(64), 0, s, base, cnt, rp,
                                   ci, ds, v, dv, nullptr, b);
            else if (join)
                hipLaunchKernelGGL((k_bsgs_w<B, false, false, K, true>), g, dim3(64), 0, s, base,
                                   cnt, rp, ci, ds, v, dv, nullptr, b);
            else
                hipLaunchKernelGGL((k_bsgs_w<B, false, false, K>), g, dim3(64), 0, s, base, cnt, rp,
                                   ci, ds, v, dv, nullptr, b);
            return ok();
        }
    }
    const dim3 g((cnt + KB - 1)/KB);
    if (upper)
        hipLaunchKernelGGL((k_sweep64<B, true, K>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci, ds, v,
                           dv, b);
    else
        hipLaunchKernelGGL((k_sweep64<B, false, K>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci, ds,
                           v, dv, b);
    return ok();
}

template <int B> struct Sw64L {
    static int run(hipStream_t s, int kind, int upper, int base, int cnt, const int *ord,
                   const int *rp, const int *ci, const int *ds, const double *v, const double *dv,
                   double *b, bool empty, bool join)
    {
        switch (kind) {
        case SW_LUSGS:
            return sweep64_launch<B, SW_LUSGS>(s, upper, base, cnt, ord, rp, ci, ds, v, dv, b, empty,
                                               join);
        case SW_BILU:
            return sweep64_launch<B, SW_BILU>(s, upper, base, cnt, ord, rp, ci, ds, v, dv, b, empty,
                                               join);
        case SW_ILU:
            if (B != 1) return UCFD_ERR_ARG;
            return sweep64_launch<1, SW_ILU>(s, upper, base, cnt, ord, rp, ci, ds, v, dv, b, empty,
                                               join);
        default:
            return UCFD_ERR_ARG;
        }
    }
};

template <int B> struct Sw32L {
    static int run(hipStream_t s, int upper, int base, int cnt, const int *ord, const int *rp,
                   const int *ci, const int *ds, const float *v, const double *dv, float *x32,
                   double *b, bool empty, bool join)
    {
        if (B > 1 && !ord) {
            const dim3 g((cnt + 64/B - 1)/(64/B));
            if (empty) {
                // no row of the level takes a block in this direction
                if (upper)
                    hipLaunchKernelGGL((k_bsgs_diag<B, true, true, SW_LUSGS>), g, dim3(64), 0, s,
                                       base, cnt, dv, x32, b);
                else
                    hipLaunchKernelGGL((k_bsgs_diag<B, false, true, SW_LUSGS>), g, dim3(64), 0, s,
                                       base, cnt, dv, x32, b);
                return ok();
            }
            if (upper)
                hipLaunchKernelGGL((k_bsgs_w<B, true, true, SW_LUSGS>), g, dim3(64), 0, s, base, cnt,
                                   rp, ci, ds, v, dv, x32, b);
            else if (join)
                hipLaunchKernelGGL((k_bsgs_w<B, false, true, SW_LUSGS, true>), g, dim3(64), 0, s,
                                   base, cnt, rp, ci, ds, v, dv, x32, b);
            else
                hipLaunchKernelGGL((k_bsgs_w<B, false, true, SW_LUSGS>), g, dim3(64), 0, s, base,
                                   cnt, rp, ci, ds, v, dv, x32, b);
            return ok();
        }
        const dim3 g((cnt + KB - 1)/KB);
        if (upper)
            hipLaunchKernelGGL((k_sweep32<B, true>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci, ds, v,
                               dv, x32, b);
        else
            hipLaunchKernelGGL((k_sweep32<B, false>), g, dim3(KB), 0, s, base, cnt, ord, rp, ci, ds,
                               v, dv, x32, b);
        return ok();
    }
};

}  // namespace

int kry_spmv_bsr(hipStream_t s, int bn, int blk, const int *rowptr, const int *colidx,
                 const double *values, double alpha, const double *x, double beta, double *y,
                 int *flag)
{
    if (bn <= 0) return UCFD_OK;
    return by_block<SpmvL>(blk, s, bn, rowptr, colidx, values, alpha, x, beta, y, flag);
}

int kry_spmv_csr(hipStream_t s, int n, const int *rowptr, const int *colidx, const double *values,
                 double alpha, const double *x, double beta, double *y, int *flag)
{
    if (n <= 0) return UCFD_OK;
    hipLaunchKernelGGL(k_spmv_csr, dim3((n + KB - 1)/KB), dim3(KB), 0, s, n, rowptr, colidx,
                       values, alpha, x, beta, y, flag);
    return ok();
}

int kry_bsgs_prepare(hipStream_t s, int bn, int blk, int64_t nnz, const int *diagslots,
                     const double *values, double *diagvalues, float *vals32, int *flag)
{
    if (bn <= 0) return UCFD_OK;
    int rc = by_block<PrepL>(blk, s, bn, diagslots, values, diagvalues, flag);
    if (rc || !vals32) return rc;
    const int64_t n = nnz*blk*blk;
    hipLaunchKernelGGL(k_to32, dim3(nblocks(n)), dim3(KB), 0, s, n, values, vals32);
    return ok();
}

int kry_ilu_factor(hipStream_t s, int scalar, int rows, int blk, int base, int cnt,
                   const int *order, const int *rowptr, const int *colidx, const int *diagslots,
                   double *values, double *diagvalues, int *flag)
{
    if (cnt <= 0) return UCFD_OK;
    return by_block<IluL>(blk, s, scalar != 0, rows != 0, base, cnt, order, rowptr, colidx,
                          diagslots, values, diagvalues, flag);
}

int kry_bsgs_sweep64(hipStream_t s, int kind, int upper, int blk, int base, int cnt,
                     const int *order, const int *rowptr, const int *colidx, const int *diagslots,
                     const double *values, const double *diagvalues, double *b, bool empty,
                     bool join)
{
    if (cnt <= 0) return UCFD_OK;
    return by_block<Sw64L>(blk, s, kind, upper, base, cnt, order, rowptr, colidx, diagslots,
                           values, diagvalues, b, empty, join);
}

int kry_bsgs_sweep32(hipStream_t s, int upper, int blk, int base, int cnt, const int *order,
                     const int *rowptr, const int *colidx, const int *diagslots,
                     const float *vals32, const double *diagvalues, float *x32, double *b,
                     bool empty, bool join)
{
    if (cnt <= 0) return UCFD_OK;
    return by_block<Sw32L>(blk, s, upper, base, cnt, order, rowptr, colidx, diagslots, vals32,
                           diagvalues, x32, b, empty, join);
}

namespace {

// partials a consumer finds per row of a reduction over n elements
int row_np(int64_t n) { return nblocks(n) <= KFUSE ? nblocks(n) : 1; }

void shorten_rows(hipStream_t s, int64_t n, double *part, int rows)
{
    if (nblocks(n) > KFUSE)
        hipLaunchKernelGGL(k_sum_rows, dim3(rows), dim3(1024), 0, s, part, nblocks(n));
}

}  // namespace

int kry_dot(hipStream_t s, int64_t n, const double *x, const double *y, double *part, double *out,
            const KryPost &h)
{
    const int nb = nblocks(n);
    hipLaunchKernelGGL(k_dot, dim3(nb), dim3(KB), 0, s, n, x, y, part);
    shorten_rows(s, n, part, 1);
    if (out) hipLaunchKernelGGL(k_sum_row, dim3(1), dim3(64), 0, s, part, row_np(n), out, h);
    return ok();
}

int kry_dot5(hipStream_t s, int64_t n, const double *rt, const double *sv, const double *t,
             double *part)
{
    hipLaunchKernelGGL(k_dot5, dim3(nblocks(n)), dim3(KB), 0, s, n, rt, sv, t, part);
    shorten_rows(s, n, part, 5);
    return ok();
}

int kry_gemvt(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv, const double *w,
              double *part)
{
    if (k <= 0 || k > 64) return UCFD_ERR_ARG;
    const int nb = nblocks(n);
    if (k <= 8)
        hipLaunchKernelGGL(k_gemvt_all<8>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, w, part);
    else if (k <= 16)
        hipLaunchKernelGGL(k_gemvt_all<16>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, w, part);
    else if (k <= 32)
        hipLaunchKernelGGL(k_gemvt_all<32>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, w, part);
    else
        for (int j0 = 0; j0 < k; j0 += 8)
            hipLaunchKernelGGL(k_gemvt8, dim3(nb), dim3(KB), 0, s, n, k, j0, V, ldv, w, part);
    shorten_rows(s, n, part, k);
    return ok();
}

int kry_gemv_gemvt(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv, double alpha,
                   const double *hpart, double *w, double *part, const KryPost &h)
{
    if (k <= 0 || k > 64) return UCFD_ERR_ARG;
    if (k > 32) {
        int rc = kry_gemv(s, n, k, V, ldv, alpha, hpart, w, nullptr, h);
        return rc ? rc : kry_gemvt(s, n, k, V, ldv, w, part);
    }
    const int nb = nblocks(n), np = row_np(n);
    if (k <= 8)
        hipLaunchKernelGGL(k_gemv_gemvt<8>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart,
                           np, w, part, h);
    else if (k <= 16)
        hipLaunchKernelGGL(k_gemv_gemvt<16>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart,
                           np, w, part, h);
    else
        hipLaunchKernelGGL(k_gemv_gemvt<32>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart,
                           np, w, part, h);
    shorten_rows(s, n, part, k);
    return ok();
}

int kry_gemv(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv, double alpha,
             const double *hpart, double *w, double *part, const KryPost &h)
{
    if (k <= 0 || k > 64) return UCFD_ERR_ARG;
    const int nb = nblocks(n), np = row_np(n);
    if (k <= 8)
        hipLaunchKernelGGL(k_gemv_r<8>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart, np,
                           w, part, h);
    else if (k <= 16)
        hipLaunchKernelGGL(k_gemv_r<16>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart, np,
                           w, part, h);
    else if (k <= 32)
        hipLaunchKernelGGL(k_gemv_r<32>, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart, np,
                           w, part, h);
    else
        hipLaunchKernelGGL(k_gemv, dim3(nb), dim3(KB), 0, s, n, k, V, ldv, alpha, hpart, np, w,
                           part, h);
    if (part) shorten_rows(s, n, part, 1);
    return ok();
}

int kry_gemv_y(hipStream_t s, int64_t n, int k, const double *V, int64_t ldv, const KryCoef &y,
               double *x)
{
    if (k <= 0 || k > 64) return UCFD_ERR_ARG;
    if (k <= 8)
        hipLaunchKernelGGL(k_gemv_y<8>, dim3(nblocks(n)), dim3(KB), 0, s, n, k, V, ldv, y, x);
    else
        hipLaunchKernelGGL(k_gemv_y<16>, dim3(nblocks(n)), dim3(KB), 0, s, n, k, V, ldv, y, x);
    return ok();
}

int kry_scale_by_inv_sqrt(hipStream_t s, int64_t n, const double *src, const double *nsq_part,
                          double *dst, double *dst2, const KryPost &h)
{
    hipLaunchKernelGGL(k_scale_isqrt, dim3(nblocks(n)), dim3(KB), 0, s, n, src, nsq_part, row_np(n),
                       dst, dst2, h);
    return ok();
}

int kry_axpy(hipStream_t s, int64_t n, double a, const double *x, double *y)
{
    hipLaunchKernelGGL(k_axpby, dim3(nblocks(n)), dim3(KB), 0, s, n, a, x, 0.0, y, 0);
    return ok();
}

int kry_axpby(hipStream_t s, int64_t n, double a, const double *x, double b, double *y)
{
    hipLaunchKernelGGL(k_axpby, dim3(nblocks(n)), dim3(KB), 0, s, n, a, x, b, y, 1);
    return ok();
}

int kry_copy(hipStream_t s, int64_t n, const double *x, double *y)
{
    hipLaunchKernelGGL(k_axpby, dim3(nblocks(n)), dim3(KB), 0, s, n, 0.0, x, 0.0, y, 2);
    return ok();
}

int kry_fill(hipStream_t s, int64_t n, double v, double *y)
{
    hipLaunchKernelGGL(k_axpby, dim3(nblocks(n)), dim3(KB), 0, s, n, v, (const double *)nullptr, 0.0,
                       y, 3);
    return ok();
}

int kry_bicg_p(hipStream_t s, int64_t n, double beta, double omega, const double *r,
               const double *v, double *p, double *pt)
{
    hipLaunchKernelGGL(k_bicg_p, dim3(nblocks(n)), dim3(KB), 0, s, n, beta, omega, r, v, p, pt);
    return ok();
}

int kry_bicg_s(hipStream_t s, int64_t n, double rho, const double *pi_part, const double *r,
               const double *v, double *sv, double *shat)
{
    hipLaunchKernelGGL(k_bicg_s, dim3(nblocks(n)), dim3(KB), 0, s, n, rho, pi_part, row_np(n),
                       r, v, sv, shat);
    return ok();
}

int kry_cast32(hipStream_t s, int64_t n, const double *a, float *b)
{
    if (n <= 0) return UCFD_OK;
    hipLaunchKernelGGL(k_cast32, dim3(nblocks(n)), dim3(KB), 0, s, n, a, b);
    return ok();
}

int kry_bicg_xr(hipStream_t s, int64_t n, double rho, const double *pi_part, const double *dots,
                const double *pt, const double *shat, const double *sv, const double *t, double *x,
                double *r, const KryPost &h)
{
    hipLaunchKernelGGL(k_bicg_xr, dim3(nblocks(n)), dim3(KB), 0, s, n, rho, pi_part, dots,
                       row_np(n), pt, shat, sv, t, x, r, h);
    return ok();
}
