// Wave-level block-row helpers shared by the block kernels (BSR SpMV, the
// block LU-SGS apply, the FlowSys block sweeps).
//
// One wave (64 lanes, one wave per workgroup) serves G = 64 / B block rows;
// lane (g, r) = (lane / B, lane % B) owns scalar row r of block row g.  A block
// is row-major, so one lane's scalar row is B contiguous values and the lanes of
// a group cover the block: with loads of several values each, a wave reads its
// rows' k-th blocks in two or three instructions.  Each lane keeps the summation
// order of its scalar row, so results equal those of a thread-per-row kernel bit
// for bit.
#pragma once

#include <hip/hip_runtime.h>

namespace ucfd {

// LDS ordering inside one wave: LDS operations of a wave execute in order,
// the fences keep the compiler from moving LDS accesses across this point.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// N consecutive values at p (aligned to one value) in the widest loads that
// cover them
typedef double wr_d2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float wr_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float wr_f2 __attribute__((ext_vector_type(2), aligned(4)));

template <int N> __device__ __forceinline__ void ld_values(const double *p, double *v)
{
#pragma unroll
    for (int q = 0; q + 2 <= N; q += 2) {
        const wr_d2 *a = (const wr_d2 *)(p + q);
        const wr_d2 t = *a;
        v[q] = t.x;
        v[q + 1] = t.y;
    }
    if (N % 2) v[N - 1] = p[N - 1];
}

template <int N> __device__ __forceinline__ void ld_values(const float *p, float *v)
{
#pragma unroll
    for (int q = 0; q + 4 <= N; q += 4) {
        const wr_f4 *a = (const wr_f4 *)(p + q);
        const wr_f4 t = *a;
        v[q] = t.x;
        v[q + 1] = t.y;
        v[q + 2] = t.z;
        v[q + 3] = t.w;
    }
    constexpr int R = N/4*4;
    if (N - R >= 2) {
        const wr_f2 *a = (const wr_f2 *)(p + R);
        const wr_f2 t = *a;
        v[R] = t.x;
        v[R + 1] = t.y;
    }
    if (N % 2) v[N - 1] = p[N - 1];
}

// one-wave workgroups remapped so that each XCD owns runs of 32 consecutive
// waves, the 8 XCDs neighbouring runs (hardware deals workgroup ids
// round-robin over the XCDs): adjacent rows share one L2 while the XCDs
// work on nearby rows (3-4 % faster block sweeps than one contiguous eighth
// per XCD).  The last incomplete group of runs keeps the identity.
__device__ __forceinline__ int wave_xcd_index()
{
    constexpr int RUN = 32;
    const int b = blockIdx.x, nblk = gridDim.x;
    const int full = nblk/(8*RUN)*(8*RUN);
    if (b >= full) return b;
    const int x = b % 8, k = b / 8;
    return (k/RUN)*(8*RUN) + x*RUN + k%RUN;
}

}  // namespace ucfd
