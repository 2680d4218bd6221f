// Adjoint of one FP64 coloured LU-SGS pass (pre + lower + upper) on a
// colour-contiguous numbering: the transposed sweeps.  The upper sweep's
// adjoint runs colours ascending, the lower sweep's colours descending; a
// cell gathers the adjoint of its already-processed neighbours through the
// face-pair map (the neighbour's face pointing back to it), in face order,
// so there are no atomics and results are deterministic.  The lower-sweep
// launch also finishes the cell's gradients with respect to rhsb, dt (via
// the pre diagonal) and fspr.  Operation order = oracle/adjoint_oracle.c.
//
// rhsbar may alias dstar: the lower-sweep adjoint reads a cell's own dstar
// before writing its rhsbar, and reads dstar only of cells in lower colours,
// which it processes later (colours descending).
#include <hip/hip_runtime.h>

#include "adjoint_internal.h"
#include "error_word.h"
#include "flux.h"

namespace {

constexpr int AB = 256;

__device__ __forceinline__ int axcd()
{
    const int b = blockIdx.x, nblk = gridDim.x;
    const int x = b % 8, k = b / 8, per = nblk / 8, rem = nblk % 8;
    return x*per + (x < rem ? x : rem) + k;
}

int ok() { return hipGetLastError() == hipSuccess ? UCFD_OK : UCFD_ERR_HIP; }

__global__ __launch_bounds__(AB) void k_pairs(int64_t N, int F, const int *__restrict__ nei,
                                              int *__restrict__ pair, int *flag)
{
    const int64_t i = (int64_t)blockIdx.x*AB + threadIdx.x;
    if (i >= N) return;
    for (int f = 0; f < F; ++f) {
        const int64_t nb = nei[f*N + i];
        int pf = -1;
        if ((uint64_t)nb >= (uint64_t)N) {
            ucfd::raise(flag, UCFD_KFLAG_INDEX);
        } else if (nb != i) {
            for (int g = 0; g < F; ++g)
                if (nei[g*N + nb] == i) { pf = g; break; }
            if (pf < 0) ucfd::raise(flag, UCFD_KFLAG_INDEX);
        }
        pair[f*N + i] = pf;
    }
}

// Both transposed sweeps run one wave per face: a workgroup serves 64 cells
// with FC waves.  Wave k loads, sums and stores row k of its cells (k, k + FC,
// ...), wave f gathers through face f; rows and face terms meet in LDS, where
// each row is summed over the faces in index order.  A face not taken
// contributes -0.0, which leaves every sum as it is.
//
// The adjoint of a cell and its pre diagonal are kept as one record of
// rec_w<ND>() doubles, gathered as 16-byte pairs: a neighbour is one or two
// cache lines instead of one per row.
//
// Bound by the gathers (a neighbour's face data lies in the caller's rows, 5
// lines besides the record).  One adjoint call, against one thread per cell
// with [var][cell] rows and a launch of its own for the diagonal: 1M tets 214
// -> 185 us on two colours, 298 -> 252 us on four, 913K hexes 241 -> 212 us,
// 64K hexes 44 -> 33 us.  With every wave holding all the cell's rows instead
// of one each, 912K hexes took 419 us (the rows' loads six times over).
template <int ND> constexpr int rec_w() { return (ND + 4) & ~1; }

typedef double ad2 __attribute__((ext_vector_type(2)));

// one face's term: coef_j (A(U; n_j)^T x_j - lam_j x_j), coef_j = -0.5 fv_j/diag_j
template <int ND>
__device__ __forceinline__ void gather(int64_t N, int64_t j, int f, const double (*U)[64],
                                       int lane, const double *__restrict__ fnv,
                                       const double *__restrict__ vfn,
                                       const double *__restrict__ fspr, const double *rec,
                                       double *term)
{
    constexpr int NV = ND + 2, W = rec_w<ND>();
    double n[ND], u[NV], v[W], jt[NV];
    const double fv = fnv[f*N + j], lam = fspr[f*N + j];
#pragma unroll
    for (int d = 0; d < ND; ++d) n[d] = vfn[((int64_t)f*ND + d)*N + j];
    const ad2 *p = (const ad2 *)(rec + j*W);
#pragma unroll
    for (int q = 0; q < W/2; ++q) {
        const ad2 t = p[q];
        v[2*q] = t.x;
        v[2*q + 1] = t.y;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) u[k] = U[k][lane];
    ucfd::ns_flux_jt<double, ND>(u, n, v, jt);
    const double coef = -0.5*fv/v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) term[k] = coef*(jt[k] - lam*v[k]);
}

// Upper sweep transposed, colour [n0, ne): rec_i = w_i + the face terms of
// earlier colours, and the cell's pre diagonal (ucfd_launch_pre's expressions).
// ANY: the colour can have such faces (not the first one).
template <int ND, int FC, bool ANY>
__global__ __launch_bounds__(64*FC) void k_adj_upper(int n0, int ne, int64_t N,
                                                     const int *__restrict__ nei,
                                                     const int *__restrict__ pair,
                                                     const double *__restrict__ fnv,
                                                     const double *__restrict__ vfn,
                                                     const double *__restrict__ fspr,
                                                     const double *__restrict__ dt, double factor,
                                                     const double *__restrict__ upts,
                                                     const double *__restrict__ dq,
                                                     const double *__restrict__ w, double *rec)
{
    constexpr int NV = ND + 2, W = rec_w<ND>(), KW = (NV + FC - 1)/FC;
    __shared__ double sU[NV][64], sterm[ANY ? FC : 1][NV][64], sdiag[FC][64];
    const int lane = threadIdx.x & 63, f = threadIdx.x >> 6;
    const int64_t i = n0 + (int64_t)axcd()*64 + lane;
    const bool act = i < ne;
    double wk[KW];
    int64_t j = 0;
    int pf = 0;
    double ti = 1.0;
    if (act) {
        if (ANY) {
            j = nei[f*N + i];
            pf = pair[f*N + i];
        }
        sdiag[f][lane] = 0.5*fspr[f*N + i]*fnv[f*N + i];
        if (f == 0) ti = dt[i];
#pragma unroll
        for (int q = 0; q < KW; ++q) {
            const int k = f + q*FC;
            if (k >= NV) continue;
            wk[q] = w[k*N + i];
            if (ANY) sU[k][lane] = upts[k*N + i] + dq[k*N + i];
        }
    }
    __syncthreads();
    if (ANY) {
        double term[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) term[k] = -0.0;
        if (act && j < n0) gather<ND>(N, j, pf, sU, lane, fnv, vfn, fspr, rec, term);
#pragma unroll
        for (int k = 0; k < NV; ++k) sterm[f][k][lane] = term[k];
        __syncthreads();
    }
    if (!act) return;
#pragma unroll
    for (int q = 0; q < KW; ++q) {
        const int k = f + q*FC;
        if (k >= NV) continue;
        double acc = wk[q];
        if (ANY) {
#pragma unroll
            for (int g = 0; g < FC; ++g) acc += sterm[ANY ? g : 0][k][lane];
        }
        rec[i*W + k] = acc;
    }
    if (f == 0) {
        const double d = 1.0/(ti*factor) + 0.0 + 0.0;
        double sd = 0.0;
#pragma unroll
        for (int g = 0; g < FC; ++g) sd += sdiag[g][lane];
        rec[i*W + NV] = d + sd;
    }
}

// Lower sweep transposed, colour [n0, ne), and the cell's gradients: rec_i +=
// the face terms of later colours, rhsbar, dtbar, and wave f the fspr gradient
// of face f.  ANY: the colour can have such faces (not the last one).
template <int ND, int FC, bool ANY>
__global__ __launch_bounds__(64*FC) void k_adj_lower(int n0, int ne, int64_t N,
                                                     const int *__restrict__ nei,
                                                     const int *__restrict__ pair,
                                                     const double *__restrict__ fnv,
                                                     const double *__restrict__ vfn,
                                                     const double *__restrict__ fspr,
                                                     const double *__restrict__ dt, double factor,
                                                     const double *__restrict__ upts,
                                                     const double *dstar,
                                                     const double *__restrict__ dq, double *rec,
                                                     double *rhsbar,
                                                     double *__restrict__ dtbar,
                                                     double *__restrict__ fsprbar)
{
    constexpr int NV = ND + 2, W = rec_w<ND>(), KW = (NV + FC - 1)/FC;
    // rows of the cells: U = upts + dstar, a = the record, acc = a + face
    // terms, e = a (dstar - dq)/diag, r = dstar/diag
    __shared__ double sU[NV][64], sa[NV][64], sacc[NV][64], se[NV][64], sr[NV][64];
    __shared__ double sterm[ANY ? FC : 1][NV][64];
    const int lane = threadIdx.x & 63, f = threadIdx.x >> 6;
    const int64_t i = n0 + (int64_t)axcd()*64 + lane;
    const bool act = i < ne;
    double qn[NV], ak[KW], di = 1.0, fv = 0.0;
    int64_t j = 0;
    int pf = 0;
    bool inner = false, later = false;
    if (act) {
        j = nei[f*N + i];
        if (ANY) pf = pair[f*N + i];
        fv = fnv[f*N + i];
        di = rec[i*W + NV];
#pragma unroll
        for (int q = 0; q < KW; ++q) {
            const int k = f + q*FC;
            if (k >= NV) continue;
            const double ds = dstar[k*N + i], qk = dq[k*N + i], a = rec[i*W + k];
            ak[q] = a;
            if (ANY) sU[k][lane] = upts[k*N + i] + ds;
            sa[k][lane] = a;
            se[k][lane] = a*((ds - qk)/di);
            sr[k][lane] = ds/di;
        }
        inner = j != i;
        later = ANY && j >= ne;
        if (inner) {
            // the neighbour's rows that the fspr gradient multiplies
            const double *from = later ? dq : dstar;
#pragma unroll
            for (int k = 0; k < NV; ++k) qn[k] = from[k*N + j];
        }
    }
    // (rhsbar may be the dstar array: the cell's dstar rows are in LDS from here
    // on, and the rows of neighbours gathered above belong to earlier colours)
    __syncthreads();
    if (ANY) {
        double term[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) term[k] = -0.0;
        if (act && inner && later)
            gather<ND>(N, j, pf, sU, lane, fnv, vfn, fspr, rec, term);
#pragma unroll
        for (int k = 0; k < NV; ++k) sterm[f][k][lane] = term[k];
        __syncthreads();
    }
    if (act) {
#pragma unroll
        for (int q = 0; q < KW; ++q) {
            const int k = f + q*FC;
            if (k >= NV) continue;
            double acc = ak[q];
            if (ANY) {
#pragma unroll
                for (int g = 0; g < FC; ++g) acc += sterm[ANY ? g : 0][k][lane];
                rec[i*W + k] = acc;
            }
            rhsbar[k*N + i] = acc/di;
            sacc[k][lane] = acc;
        }
    }
    __syncthreads();
    if (!act) return;
    double dgb = 0.0, s = 0.0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double acc = sacc[k][lane];
        dgb += se[k][lane] - acc*sr[k][lane];
        if (inner) s += (later ? sa[k][lane] : acc)*qn[k];
    }
    if (f == 0) {
        const double t = dt[i];
        dtbar[i] = -dgb/(t*t*factor);
    }
    double val = dgb*0.5*fv;
    if (inner) val += 0.5*fv*s/di;
    fsprbar[f*N + i] = val;
}

template <int ND, int FC>
int launch(hipStream_t s, int lower, int n0, int ne, int64_t N, const int *nei, const int *pair,
           const double *fnv, const double *vfn, const double *fspr, const double *dt,
           double factor, const double *upts, const double *dstar, const double *dq,
           const double *w, double *rec, double *rhsbar, double *dtbar, double *fsprbar)
{
    const dim3 g((unsigned)((ne - n0 + 63)/64)), b(64*FC);
#define LO(ANY) hipLaunchKernelGGL((k_adj_lower<ND, FC, ANY>), g, b, 0, s, n0, ne, N, nei, pair, \
                                   fnv, vfn, fspr, dt, factor, upts, dstar, dq, rec, rhsbar,     \
                                   dtbar, fsprbar)
#define UP(ANY) hipLaunchKernelGGL((k_adj_upper<ND, FC, ANY>), g, b, 0, s, n0, ne, N, nei, pair, \
                                   fnv, vfn, fspr, dt, factor, upts, dq, w, rec)
    if (lower) { if (ne < N) LO(true); else LO(false); }
    else { if (n0 > 0) UP(true); else UP(false); }
#undef LO
#undef UP
    return ok();
}

}  // namespace

int adj_launch_pairs(hipStream_t s, int64_t N, int F, const int *nei, int *pair, int *flag)
{
    if (N <= 0) return UCFD_OK;
    hipLaunchKernelGGL(k_pairs, dim3((unsigned)((N + AB - 1)/AB)), dim3(AB), 0, s, N, F, nei, pair,
                       flag);
    return ok();
}

size_t adj_rec_doubles(int ndims) { return ndims == 3 ? rec_w<3>() : rec_w<2>(); }

int adj_launch_colour(hipStream_t s, int lower, int n0, int ne, int64_t N, int nface, int ndims,
                      const int *nei, const int *pair, const double *fnv, const double *vfn,
                      const double *fspr, const double *dt, double factor, const double *upts,
                      const double *dstar, const double *dq, const double *w, double *rec,
                      double *rhsbar, double *dtbar, double *fsprbar)
{
    if (ne <= n0) return UCFD_OK;
#define ADJ_CASE(D, FC)                                                                          \
    if (ndims == D && nface == FC)                                                               \
        return launch<D, FC>(s, lower, n0, ne, N, nei, pair, fnv, vfn, fspr, dt, factor, upts,  \
                             dstar, dq, w, rec, rhsbar, dtbar, fsprbar);
    ADJ_CASE(3, 4)
    ADJ_CASE(3, 6)
    ADJ_CASE(3, 5)
    ADJ_CASE(2, 3)
    ADJ_CASE(2, 4)
#undef ADJ_CASE
    return UCFD_ERR_ARG;
}
