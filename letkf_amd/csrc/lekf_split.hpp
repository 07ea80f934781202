// lekf_split.hpp -- the workspace record of the solves that read a point's Gram from
// global memory (k > 32), and what their kernels share.
#pragma once
#include "lekf_dev.hpp"

namespace {

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Adaptive inflation update (common_letkf.f90:218-239)
__device__ __forceinline__ double adaptive_alpha(double alpha, double p1, double p2, double p3)
{
    const double p4 = (p1 - p3) / p2 - alpha;
    const double qv = (alpha * p2 + p3) / p2;
    const double so = 2.0 / p3 * (qv * qv);
    const double sb2 = 0.04 * 0.04;
    return alpha + sb2 / (so + sb2) * p4;
}

// workspace record of one point: C (k x k, row-major), b (k), sum w d^2, P3
__host__ __device__ inline long gram_stride(int kmax)
{
    return ((long)kmax * kmax + kmax + 2 + 1) & ~1L;
}

// split-record flag: the mixed-precision pass found C ill-conditioned and put
// the point on the redo list, whose points a second pass solves again from an
// FP64 Gram after the launch's last sub-batch
constexpr int kSplitRedo = 16;

// split-record flag: the point is left to lekf_eig_fix_kernel (its rotation stream
// overflowed, or its condition number is past the rational form's tables), which finds
// its slot in flist (flist[0] entries from flist[1])
constexpr int kSplitOverflow = 8;
__device__ inline void split_flag_slot(int* flist, long slot)
{
    flist[1 + atomicAdd(flist, 1)] = (int)slot;
}

// Flat point of slot `slot` of a split kernel: pass 0 the sub-batch's own
// (gp0 + slot, nb slots), pass 1 the redo list's (rlist[0] entries from
// rlist[1], of which the first nb were written: the count goes on past the
// list's capacity); false past the end.
__device__ inline bool split_slot_point(long slot, long gp0, long nb, int pass,
                                        const int* rlist, long& gp)
{
    if (pass) {
        if (slot >= nb || slot >= rlist[0]) return false;
        gp = rlist[1 + slot];
        return true;
    }
    gp = gp0 + slot;
    return slot < nb;
}

// The plain solve (lekf_trf.hip): offsets in a point's record
struct TrfRec {
    long d, e, tau, mean, sc, z, v;  // offsets in the point's record
};
constexpr int kTrfSc = 4;  // sc: m, table level, trace of C

__host__ __device__ inline TrfRec trf_rec(int kmax)
{
    TrfRec S;
    S.d = gram_stride(kmax) + 2;  // after the flag
    S.e = S.d + kmax;
    S.tau = S.e + kmax;
    S.mean = S.tau + kmax;
    S.sc = S.mean + LEKF_NVMAX + 1;
    S.z = S.sc + kTrfSc;
    S.v = S.z + (long)(LEKF_NVMAX + 1) * kmax;
    return S;
}
__host__ __device__ inline long trf_stride(int kmax)
{
    return (trf_rec(kmax).v + (long)kmax * kmax + 1) & ~1L;
}

}  // namespace

// the plain solve of a sub-batch of nb slots (lekf_trf.hip)
hipError_t lekf_trf_launch(long nb, hipStream_t st, const LekfJob* djobs, int njobs, long g0,
                           double* ws, long gs, int nvmax, int kmax, int pass, int mode,
                           double kthr, int* rlist, long lcap, int* flist);
