// Sequential sweeps of the serial legacy API (serial_ns_*, serial_rans_* and
// their two-array forms): cell i after every neighbour before it (lower) or
// after it (upper), as src/lusgs/lusgs.c:157-321 visits them, in one launch.
//
// Cells are taken in sweep order, KB consecutive ones by a workgroup, one to a
// lane, so the geometry of a wave is met in whole lines.  A lane waits for the
// solution of the neighbours that it takes and publishes its own: in LDS for its
// workgroup, in pub (device memory, [rows][N]) for the others.  A word of both
// holds kUnset until the value is there, so the wait for a value is the load of
// it, and no flag, fence or barrier orders two cells; values are loaded and
// stored as relaxed atomics of workgroup / agent scope.  A value whose bits are
// kUnset (one NaN of 2^52) is published as the next NaN.
//
// Every wait ends: a cell takes only neighbours earlier in the sweep, and a
// workgroup draws its cells by a ticket when it starts, so the earliest unfinished
// cell is always ready and belongs to a workgroup that runs, or to the next one to
// start once those before it have ended.  No lane stops while another lane of its
// wave can go on.  A wave that ends after a long wait counts itself in ctl->ended, so
// a wait in a sweep that goes on is told from one in a sweep that does not: kPolls
// idle rounds (0.2 us each or more: a second) without a change there raise
// UCFD_KFLAG_STALL, and the launch drains.  The first unfinished wave ends after at
// most 64 hops, 0.3 ms; a wave may wait for all that the chip holds, 0.8 s in a chain
// of 200K cells of k_serial_any.
//
// What bounds it is the longest chain of cells; a hop costs a round of the loop
// below, about 2 us (the loads of the awaited words, up to KS fluxes, the divisions
// of the update).  A launch per dependency level cost 10 us a level, and the levels
// were found on the host, from a table that was hashed at every call and copied back
// when another one came.  A lower and an upper sweep with the update, a table
// of another address at each call: 50K hexes 5.30 -> 0.56 ms, 197K hexes 11.1 ->
// 1.2, 8K tets 0.74 -> 0.24, 197K tets 4.8 -> 0.63, 1.3M tets 19 -> 1.3; with the
// same table at every call 1.3M hexes 17.7 -> 7.9, 1.3M tets 5.5 -> 1.3.
// On numberings of few levels the launch per level was all but as good: one lower
// sweep, two levels, 91K hexes 150 -> 32 us, 2.0M 284 -> 224, 1.3M tets 210 -> 130,
// 5.3M 425 -> 470 (the 212 MB of pub, set and written); four levels 541 -> 537.
// On the 50K hexes: all faces in slots (256 VGPRs and more, one wave a SIMD) with
// the flux of u inside the chain 0.92 ms; memory asked only in rounds in which
// nothing moves inside the workgroup 0.75, or while up to four rounds inside run
// 0.90; one flux a round for whichever slot is ready 0.92; two slots 0.90; 128
// cells a workgroup 0.79 and 512 0.84 against 0.75.
#include "error_word.h"
#include "flux.h"
#include "ucfd_internal.h"

namespace {

constexpr int KB = 256;   // cells of a workgroup
constexpr int KS = 3;     // faces of a cell that wait at the same time
constexpr int kPolls = 1 << 22;
typedef unsigned long long word;
constexpr word kUnset = 0xFFF8A5C35A3C0F1Eull;

// behind the words of pub
struct Control {
    word ticket;            // workgroups started
    unsigned stall, ended;  // a wave has given up; waves that waited long and ended
};
constexpr int kControl = sizeof(Control)/sizeof(word);

__global__ __launch_bounds__(256) void k_unset(int64_t n, word *pub)
{
    const int64_t st = (int64_t)gridDim.x*256;
    for (int64_t k = (int64_t)blockIdx.x*256 + threadIdx.x; k < n + kControl; k += st)
        pub[k] = k < n ? kUnset : 0ull;
}

__device__ __forceinline__ word to_word(double v)
{
    const word w = (word)__double_as_longlong(v);
    return w == kUnset ? kUnset + 1 : w;
}

// A face's term of the sum over the taken faces: everything that does not wait
// for the neighbour's solution is loaded before the wait.  NT == 0: the flow rows
// (lusgs.c:157-257), else NT turbulence rows behind them (lusgs.c:274-321).
template <int ND, int NT> struct Term {
    static constexpr int R = ND + 2, NV = ND + 2;
    double u[NV], f0[NV], nf[ND], fv, lam;
    __device__ __forceinline__ void load(int64_t N, int64_t i, int f, int64_t nb, const double *fnv,
                                         const double *vfn, const double *upts,
                                         const double *fspr)
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) u[k] = upts[k*N + nb];
#pragma unroll
        for (int d = 0; d < ND; ++d) nf[d] = vfn[(f*ND + d)*N + i];
        fv = fnv[f*N + i];
        lam = fspr[f*N + i];
        ucfd::ns_flux<double, ND>(u, nf, f0);
    }
    __device__ __forceinline__ void eval(const double *du, double *t) const
    {
        double up[NV], dfj[NV];   // ucfd::diff_flux with the flux of u formed before
#pragma unroll
        for (int k = 0; k < NV; ++k) up[k] = du[k] + u[k];
        ucfd::ns_flux<double, ND>(up, nf, dfj);
#pragma unroll
        for (int k = 0; k < NV; ++k) t[k] = (dfj[k] - f0[k] - lam*du[k])*fv;
    }
};

template <int ND> struct TurbBase {
    double th, fv, lam;
    __device__ __forceinline__ void load(int64_t N, int64_t i, int f, int64_t nb, const double *fnv,
                                         const double *vfn, const double *upts,
                                         const double *fspr)
    {
        th = 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) th += upts[(d + 1)*N + nb]*vfn[(f*ND + d)*N + i];
        th /= upts[nb];
        fv = fnv[f*N + i];
        lam = fspr[f*N + i];
    }
};

template <int ND, int NT> struct TurbTerm : TurbBase<ND> {
    static constexpr int R = NT;
    double ut[NT];
    __device__ __forceinline__ void load(int64_t N, int64_t i, int f, int64_t nb, const double *fnv,
                                         const double *vfn, const double *upts,
                                         const double *fspr)
    {
#pragma unroll
        for (int k = 0; k < NT; ++k) ut[k] = upts[(ND + 2 + k)*N + nb];
        TurbBase<ND>::load(N, i, f, nb, fnv, vfn, upts, fspr);
    }
    __device__ __forceinline__ void eval(const double *du, double *t) const
    {
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const double dfj = (du[k] + ut[k])*this->th - ut[k]*this->th;
            t[k] = (dfj - this->lam*du[k])*this->fv;
        }
    }
};
template <int ND> struct Term<ND, 1> : TurbTerm<ND, 1> {};
template <int ND> struct Term<ND, 2> : TurbTerm<ND, 2> {};

// the ticket of the workgroup: its place in the sweep
__device__ __forceinline__ int draw(word *ticket, int *sb)
{
    if (threadIdx.x == 0)
        *sb = (int)__hip_atomic_fetch_add(ticket, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return *sb;
}

// The idle rounds of a wave since the launch last made progress
struct Idle {
    int rounds = 0;
    unsigned ended = 0;
    __device__ __forceinline__ bool long_wait() const { return rounds >= 1024 || ended; }
    // after a round without progress: whether to give up
    __device__ __forceinline__ bool give_up(Control *ctl, int *flag)
    {
        if (++rounds & 1023) return false;
        if (__hip_atomic_load(&ctl->stall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return true;
        const unsigned e = __hip_atomic_load(&ctl->ended, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (e != ended) {
            ended = e;
            rounds = 0;
        }
        if (rounds < kPolls) return false;
        ucfd::raise(flag, UCFD_KFLAG_STALL);
        __hip_atomic_store(&ctl->stall, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
};

// By a wave whose cells are all done, if it ever had to wait for long: those that did
// not end within a millisecond, and counting every wave in one word cost 10 ns each
// (5.3M cells in two levels 0.47 -> 1.27 ms).
__device__ __forceinline__ void count_end(const Idle &idle, Control *ctl)
{
    if (idle.long_wait() && (threadIdx.x & 63) == 0)
        __hip_atomic_fetch_add(&ctl->ended, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int R> struct Chain {   // one lane's view of the published values
    word (*lds)[KB], *pub;
    int64_t N, q0;                // q0: the workgroup's first place in the sweep
    __device__ __forceinline__ bool inside(int64_t q) const { return q >= q0; }
    __device__ __forceinline__ void fetch_in(int64_t q, word *v) const
    {
#pragma unroll
        for (int k = 0; k < R; ++k)
            v[k] = __hip_atomic_load(&lds[k][q - q0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void fetch_out(int64_t q, word *v) const
    {
#pragma unroll
        for (int k = 0; k < R; ++k)
            v[k] = __hip_atomic_load(pub + k*N + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void publish(int64_t q, int k, double v) const
    {
        const word w = to_word(v);
        __hip_atomic_store(&lds[k][q - q0], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_store(pub + k*N + q, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ static __forceinline__ bool set(const word *v)
    {
        bool s = true;
#pragma unroll
        for (int k = 0; k < R; ++k) s = s && v[k] != kUnset;
        return s;
    }
};

// FC faces known at compile time: the taken faces of a cell wait KS at a time side
// by side, in face order, with what they need besides in registers.
template <int DIR, int ND, int NT, int FC>
__global__ __launch_bounds__(KB) void k_serial(int N, const int *__restrict__ nei,
                                               const double *__restrict__ fnv,
                                               const double *__restrict__ vfn,
                                               const double *__restrict__ upts, const double *in,
                                               double *out, const double *__restrict__ diag,
                                               const double *__restrict__ fspr, word *pub, int *flag)
{
    typedef Term<ND, NT> T;
    constexpr int R = T::R, K0 = NT ? ND + 2 : 0;
    __shared__ word lds[R][KB];
    __shared__ int sb;
#pragma unroll
    for (int k = 0; k < R; ++k) lds[k][threadIdx.x] = kUnset;
    Control *ctl = (Control *)(pub + (int64_t)R*N);
    const int b = draw(&ctl->ticket, &sb);
    const Chain<R> C{lds, pub, N, (int64_t)b*KB};
    const int64_t q = C.q0 + threadIdx.x, i = DIR == 0 ? q : N - 1 - q;
    bool wait = q < N;
    int nb[FC], rest = 0;      // taken faces not yet in a slot
    int nq[KS], pend = 0;      // a slot's place in the sweep; slots that wait
    T face[KS];
    double dg = 1.0, xin[R], df[R], t[KS][R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        df[k] = 0.0;
#pragma unroll
        for (int s = 0; s < KS; ++s) t[s][k] = 0.0;
    }
    if (wait) {
#pragma unroll
        for (int f = 0; f < FC; ++f) nb[f] = nei[(int64_t)f*N + i];
        dg = diag[i];
#pragma unroll
        for (int k = 0; k < R; ++k) xin[k] = in[(int64_t)(K0 + k)*N + i];
#pragma unroll
        for (int f = 0; f < FC; ++f) {
            if ((unsigned)nb[f] >= (unsigned)N) {
                ucfd::raise(flag, UCFD_KFLAG_INDEX);
                continue;
            }
            if ((DIR == 0 ? nb[f] : N - 1 - nb[f]) < q) rest |= 1 << f;
        }
    }
    Idle idle;
    while (__any(wait)) {
        if (wait && pend == 0 && rest) {
#pragma unroll
            for (int s = 0; s < KS; ++s) {
#pragma unroll
                for (int k = 0; k < R; ++k) t[s][k] = 0.0;
                if (!rest) continue;
                const int f = __builtin_ctz(rest);
                rest &= rest - 1;
                int n = nb[0];
#pragma unroll
                for (int g = 1; g < FC; ++g) n = f == g ? nb[g] : n;
                nq[s] = DIR == 0 ? n : N - 1 - n;
                pend |= 1 << s;
                face[s].load(N, i, f, n, fnv, vfn, upts, fspr);
            }
        }
        const int before = pend;
        word v[KS][R];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            v[s][0] = kUnset;
            if (!(pend >> s & 1)) continue;
            if (C.inside(nq[s])) C.fetch_in(nq[s], v[s]);
            else C.fetch_out(nq[s], v[s]);
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (!(pend >> s & 1) || v[s][0] == kUnset || !C.set(v[s])) continue;
            double du[R];
#pragma unroll
            for (int k = 0; k < R; ++k) du[k] = __longlong_as_double((long long)v[s][k]);
            face[s].eval(du, t[s]);
            pend &= ~(1 << s);
        }
        bool done = false;
        if (wait && pend == 0) {
            // an empty slot adds +0.0 to a sum that is never -0.0
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int k = 0; k < R; ++k) df[k] += t[s][k];
            done = !rest;
        }
        if (done) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const double x = DIR == 0 ? (xin[k] - 0.5*df[k])/dg : xin[k] - (0.5*df[k]/dg);
                C.publish(q, k, x);
                out[(int64_t)(K0 + k)*N + i] = x;
            }
            wait = false;
        }
        if (!__any(before != pend || done) && idle.give_up(ctl, flag)) return;
    }
    count_end(idle, ctl);
}

// Any face count: a lane takes its faces one after the other.
template <int DIR, int ND>
__global__ __launch_bounds__(KB) void k_serial_any(int N, int nface, const int *__restrict__ nei,
                                                   const double *__restrict__ fnv,
                                                   const double *__restrict__ vfn,
                                                   const double *__restrict__ upts,
                                                   const double *in, double *out,
                                                   const double *__restrict__ diag,
                                                   const double *__restrict__ fspr, word *pub,
                                                   int *flag)
{
    typedef Term<ND, 0> T;
    constexpr int R = T::R;
    __shared__ word lds[R][KB];
    __shared__ int sb;
#pragma unroll
    for (int k = 0; k < R; ++k) lds[k][threadIdx.x] = kUnset;
    Control *ctl = (Control *)(pub + (int64_t)R*N);
    const int b = draw(&ctl->ticket, &sb);
    const Chain<R> C{lds, pub, N, (int64_t)b*KB};
    const int64_t q = C.q0 + threadIdx.x, i = DIR == 0 ? q : N - 1 - q;
    bool wait = q < N;
    int f = -1;
    int64_t nq = 0;
    T face;
    double df[R];
#pragma unroll
    for (int k = 0; k < R; ++k) df[k] = 0.0;
    auto next = [&] {   // the next taken face, or nface
        while (++f < nface) {
            const int nb = nei[(int64_t)f*N + i];
            if ((unsigned)nb >= (unsigned)N) {
                ucfd::raise(flag, UCFD_KFLAG_INDEX);
                continue;
            }
            nq = DIR == 0 ? nb : N - 1 - nb;
            if (nq < q) {
                face.load(N, i, f, nb, fnv, vfn, upts, fspr);
                return;
            }
        }
    };
    if (wait) next();
    Idle idle;
    while (__any(wait)) {
        bool got = false;
        if (wait && f < nface) {
            word v[R];
            if (C.inside(nq)) C.fetch_in(nq, v);
            else C.fetch_out(nq, v);
            if (C.set(v)) {
                double du[R], t[R];
#pragma unroll
                for (int k = 0; k < R; ++k) du[k] = __longlong_as_double((long long)v[k]);
                face.eval(du, t);
#pragma unroll
                for (int k = 0; k < R; ++k) df[k] += t[k];
                got = true;
                next();
            }
        }
        if (wait && f >= nface) {
            const double dg = diag[i];
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const double xi = in[(int64_t)k*N + i];
                const double x = DIR == 0 ? (xi - 0.5*df[k])/dg : xi - (0.5*df[k]/dg);
                C.publish(q, k, x);
                out[(int64_t)k*N + i] = x;
            }
            wait = false;
            got = true;
        }
        if (!__any(got) && idle.give_up(ctl, flag)) return;
    }
    count_end(idle, ctl);
}

}  // namespace

size_t ucfd_serial_scratch(int neles, int rows)
{
    return ((size_t)neles*(size_t)rows + kControl)*sizeof(word);
}

int ucfd_launch_serial(hipStream_t s, int dir, int neles, int nface, int ndims, int nt,
                       const int *nei, const double *fnorm_vol, const double *vec_fnorm,
                       const double *upts, const double *in, double *out, const double *diag,
                       const double *fspr, void *scratch, int *flag)
{
    if (neles <= 0) return UCFD_OK;
    if ((ndims != 2 && ndims != 3) || nt < 0 || nt > 2) return UCFD_ERR_ARG;
    word *pub = (word *)scratch;
    const int64_t n = (int64_t)neles*(nt ? nt : ndims + 2);
    const int64_t fb = (n + kControl + 255)/256;
    hipLaunchKernelGGL(k_unset, dim3((unsigned)(fb > 4096 ? 4096 : fb)), dim3(256), 0, s, n, pub);
    const dim3 g((unsigned)(((int64_t)neles + KB - 1)/KB)), b(KB);
#define SER(DIR, ND, NT, FC) \
    hipLaunchKernelGGL((k_serial<DIR, ND, NT, FC>), g, b, 0, s, neles, nei, fnorm_vol, vec_fnorm, \
                       upts, in, out, diag, fspr, pub, flag)
#define SER_ANY(DIR, ND) \
    hipLaunchKernelGGL((k_serial_any<DIR, ND>), g, b, 0, s, neles, nface, nei, fnorm_vol, \
                       vec_fnorm, upts, in, out, diag, fspr, pub, flag)
#define SER_F(DIR, ND, NT) do { \
    if (nface == 3) SER(DIR, ND, NT, 3); \
    else if (nface == 4) SER(DIR, ND, NT, 4); \
    else if (nface == 6) SER(DIR, ND, NT, 6); \
    else if (NT) return UCFD_ERR_ARG; \
    else SER_ANY(DIR, ND); } while (0)
#define SER_T(DIR, ND) do { \
    if (nt == 0) SER_F(DIR, ND, 0); \
    else if (nt == 1) SER_F(DIR, ND, 1); \
    else SER_F(DIR, ND, 2); } while (0)
    if (dir == 0 && ndims == 3) SER_T(0, 3);
    else if (dir == 0) SER_T(0, 2);
    else if (ndims == 3) SER_T(1, 3);
    else SER_T(1, 2);
#undef SER_T
#undef SER_F
#undef SER_ANY
#undef SER
    return hipGetLastError() == hipSuccess ? UCFD_OK : UCFD_ERR_HIP;
}
