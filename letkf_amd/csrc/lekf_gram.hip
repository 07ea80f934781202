// lekf_gram.hip -- Gram of each point's local obs, 32 < k <= LEKF_KSPLIT (gfx950).
//
// W waves per point; wave w takes every W-th chunk of 64 local obs, and the partial
// Grams are summed in LDS in wave order (deterministic for a given W), then written to
// the point's workspace record.  The FP64 form is bound by issue: its matrix
// instructions (busy 70% of the time at 256 x 256 x 60, k = 50), and the vector
// instructions that fetch and scale the rows, which do not run beside them.  128 x 128 x
// 60 points, k = 50: 203 ms with the columns rounded up to whole 16-column tiles, 147 ms
// with tiles and strips; 192 x 94 x 64 global grid, k = 40: 37 -> 33 ms.  Memory does not
// show: with every row read from a few hot lines it takes 141 ms, and ordering the
// workgroups so that an XCD's points share their rows in L2 left it at 147 ms.
#include "lekf_ktime.hpp"
#include "lekf_gram.hpp"
#include "lekf_split.hpp"

namespace {

// The point of a workgroup, or false if it has nothing to do
struct GramPoint {
    const LekfJob* J;
    int b, k, p;
    long slot, off;
};
__device__ __forceinline__ bool gram_point(const LekfJob* jobs, int njobs, long gp0,
                                           const int* rlist, int* zlist, int* flist, GramPoint& P)
{
    P.slot = blockIdx.x;
    // before any kernel adds to them: the launch's first sub-batch empties the redo list,
    // every one the list of flagged slots
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (zlist) zlist[0] = 0;
        flist[0] = 0;
    }
    long gp = gp0 + P.slot;
    if (rlist) {  // FP64 pass of a split launch: slot i holds the redo list's i-th point
        if (P.slot >= rlist[0]) return false;
        gp = rlist[1 + P.slot];
    }
    P.J = jobs + lekf_job_of(jobs, njobs, gp);
    P.b = (int)(gp - P.J->pt_begin + P.J->pt0);
    P.k = P.J->k;
    P.off = P.J->loc_off[P.b];
    P.p = P.J->loc_cnt ? P.J->loc_cnt[P.b] : (int)(P.J->loc_off[P.b + 1] - P.off);
    return P.p > 0;
}

// LDS of a workgroup: C (k x k, leading dimension k + 1), b, then [0] sum w d^2,
// [4 + w] P3 of wave w
constexpr size_t gram_lds_doubles(int kmax, int W)
{
    return (size_t)kmax * (kmax + 1) + kmax + 4 + W;
}

// C, b and the sums of the workgroup's LDS to the point's record
template <int W>
__device__ __forceinline__ void gram_out(const double* A, const double* B, double* sc, double p3,
                                         int k, double* out)
{
    const int tid = threadIdx.x, lane = tid & (LEKF_WAVE - 1), wv = tid / LEKF_WAVE;
    const int lda = k + 1;
    p3 = wave_sum(p3);
    if (lane == 0) sc[4 + wv] = p3;
    __syncthreads();
    for (int t = tid; t < k * k; t += 64 * W) {
        const int i = t / k, j = t - i * k;
        out[t] = A[i * lda + j];
    }
    for (int i = tid; i < k; i += 64 * W) out[(size_t)k * k + i] = B[i];
    if (tid == 0) {
        double s = sc[4];
        for (int w = 1; w < W; ++w) s += sc[4 + w];
        out[(size_t)k * k + k] = sc[0];
        out[(size_t)k * k + k + 1] = s;
    }
}

// FP64: the columns in tiles and strips (lekf_gram.hpp).  Registers: the accumulators,
// two pairs of row sets, and what the loop keeps
constexpr int gram_f64_waves(int ntf, int ns)
{
    const int t = 4 * ntf + ns;
    return t <= 12 ? 4 : t <= 16 ? 3 : t < 22 ? 2 : 1;
}

template <int NTF, int NS, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(gram_f64_waves(NTF, NS))))
void lekf_gram_f64_kernel(const LekfJob* __restrict__ jobs, int njobs, long gp0,
                          double* __restrict__ ws, long gstride, const int* __restrict__ rlist,
                          int* __restrict__ zlist, int* __restrict__ flist)
{
    extern __shared__ double smem[];
    GramPoint P;
    if (!gram_point(jobs, njobs, gp0, rlist, zlist, flist, P)) return;
    if (gram_ntf(P.k) != NTF || gram_ns(P.k) != NS) return;  // another launch's
    const LekfJob& J = *P.J;
    const int lane = threadIdx.x & (LEKF_WAVE - 1), wv = threadIdx.x / LEKF_WAVE;
    const int k = P.k, lda = k + 1;
    double* A = smem;
    double* B = A + (size_t)k * lda;
    double* sc = B + k;
    double p3 = 0.0;
    GramAcc<NTF, NS> G;
#pragma unroll
    for (int a = 0; a < GramAcc<NTF, NS>::NT; ++a) G.t[a] = lekf_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < NTF * NS + NS * (NS + 1) / 2; ++a) G.s[a] = 0.0;
    const GramIn I = gram_in(J, P.off, P.p);
    if (I.y_sm == 1 && I.y_so >= 0 && I.y_so < (1L << 29))
        gram_strips<NTF, NS, true>(I, lane, G, p3, wv, W);
    else
        gram_strips<NTF, NS, false>(I, lane, G, p3, wv, W);
    for (int w = 0; w < W; ++w) {
        if (wv == w) store_strips<NTF, NS>(G, k, lda, lane, A, B, &sc[0], w > 0);
        __syncthreads();
    }
    gram_out<W>(A, B, sc, p3, k, ws + P.slot * gstride);
}

// FP32 (MODE 1) and split-BF16x3 (MODE 2) on NT 16-column tiles.  FP32 with 4 x 4 tiles
// takes 188 registers unless held to three waves' budget (which it fits unspilled)
constexpr int gram_waves_per_simd(int nt, int mode)
{
    return (nt == 4 && mode == 1) ? 3 : (nt == 3 && mode == 1) ? 4 : 1;
}

template <int NT, int MODE, int W>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(gram_waves_per_simd(NT, MODE))))
void lekf_gram_kernel(const LekfJob* __restrict__ jobs, int njobs, long gp0,
                      double* __restrict__ ws, long gstride, const int* __restrict__ rlist,
                      int* __restrict__ zlist, int* __restrict__ flist)
{
    extern __shared__ double smem[];
    GramPoint P;
    if (!gram_point(jobs, njobs, gp0, rlist, zlist, flist, P)) return;
    if ((P.k + 16) / 16 != NT) return;  // another launch's
    const LekfJob& J = *P.J;
    const int lane = threadIdx.x & (LEKF_WAVE - 1), wv = threadIdx.x / LEKF_WAVE;
    const int k = P.k, lda = k + 1;
    const GramIn I = gram_in(J, P.off, P.p);
    double* A = smem;
    double* B = A + (size_t)k * lda;
    double* sc = B + k;
    double p3 = 0.0;
    lekf_f4 acc[NT * (NT + 1) / 2];
#pragma unroll
    for (int a = 0; a < NT * (NT + 1) / 2; ++a) acc[a] = lekf_f4{0.f, 0.f, 0.f, 0.f};
    if (MODE == 1) {
        lekf_d4 accd[NT * (NT + 1) / 2];
#pragma unroll
        for (int a = 0; a < NT * (NT + 1) / 2; ++a) accd[a] = lekf_d4{0.0, 0.0, 0.0, 0.0};
        gram_f32<NT>(I, lane, acc, accd, p3, wv, W);
        for (int w = 0; w < W; ++w) {
            if (wv == w) store_gram<NT, false>(accd, k, lda, lane, A, B, &sc[0], w > 0);
            __syncthreads();
        }
    } else {
        gram_bf16x3<NT>(I, lane, acc, p3, wv, W);
        for (int w = 0; w < W; ++w) {
            if (wv == w) store_gram<NT, false>(acc, k, lda, lane, A, B, &sc[0], w > 0);
            __syncthreads();
        }
    }
    gram_out<W>(A, B, sc, p3, k, ws + P.slot * gstride);
}

struct GramLaunch {
    int W;
    size_t lds;
    unsigned nb;
    hipStream_t st;
    const LekfJob* djobs;
    int njobs;
    long g0;
    double* ws;
    long gs;
    const int* rlist;
    int* zlist;
    int* flist;
};
using GramKernel = void (*)(const LekfJob*, int, long, double*, long, const int*, int*, int*);

// the form of a kernel for the waves asked for
void gram_go(GramKernel w2, GramKernel w4, GramKernel w8, const GramLaunch& G)
{
    KTime kt(G.rlist ? "redo_gram" : "gram", G.st);
    const int W = G.W == 2 || G.W == 8 ? G.W : 4;
    hipLaunchKernelGGL(W == 2 ? w2 : W == 8 ? w8 : w4, dim3(G.nb), dim3(64 * W), G.lds, G.st,
                       G.djobs, G.njobs, G.g0, G.ws, G.gs, G.rlist, G.zlist, G.flist);
}

template <int NTF, int NS>
void gram_f64_go(int cuts, const GramLaunch& G)
{
    if (cuts >> gram_cut(NTF, NS) & 1)
        gram_go(lekf_gram_f64_kernel<NTF, NS, 2>, lekf_gram_f64_kernel<NTF, NS, 4>,
                lekf_gram_f64_kernel<NTF, NS, 8>, G);
}

template <int NT, int MODE>
void gram_mixed_go(int cuts, const GramLaunch& G)
{
    // NT tiles: NT whole ones, or strips after NT - 1
    const int of = 1 << gram_cut(NT, 0) | 1 << gram_cut(NT - 1, 1) | 1 << gram_cut(NT - 1, 2);
    if (cuts & of)
        gram_go(lekf_gram_kernel<NT, MODE, 2>, lekf_gram_kernel<NT, MODE, 4>,
                lekf_gram_kernel<NT, MODE, 8>, G);
}

}  // namespace

// The jobs of a launch may have several cuts: each has its own kernel, whose workgroups
// leave the other points alone.  (Splitting the batch by cut instead repeats the solve's
// other kernels too, whose latencies do not shrink with it: 15 trans jobs of k = 33..47,
// two points each, take 1.7 ms in one launch and took 3.7 ms split.)
hipError_t lekf_gram_launch(int mode, int W, int kmax, int outs, long nb, hipStream_t st,
                            const LekfJob* djobs, int njobs, long g0, double* ws, long gs,
                            const int* rlist, int* zlist, int* flist)
{
    const GramLaunch G{W, gram_lds_doubles(kmax, W) * sizeof(double), (unsigned)nb, st, djobs,
                       njobs, g0, ws, gs, rlist, zlist, flist};
    const int cuts = outs >> LEKF_OUT_CUT0;
    if (cuts <= 0 || cuts >> kGramCuts) return hipErrorInvalidValue;
    switch (mode) {
    case 0:
        gram_f64_go<2, 1>(cuts, G);
        gram_f64_go<2, 2>(cuts, G);
        gram_f64_go<3, 0>(cuts, G);
        gram_f64_go<3, 1>(cuts, G);
        gram_f64_go<3, 2>(cuts, G);
        gram_f64_go<4, 0>(cuts, G);
        gram_f64_go<4, 1>(cuts, G);
        gram_f64_go<4, 2>(cuts, G);
        gram_f64_go<5, 0>(cuts, G);
        gram_f64_go<5, 1>(cuts, G);
        gram_f64_go<5, 2>(cuts, G);
        gram_f64_go<6, 0>(cuts, G);
        break;
    case 1:
        gram_mixed_go<3, 1>(cuts, G);
        gram_mixed_go<4, 1>(cuts, G);
        gram_mixed_go<5, 1>(cuts, G);
        gram_mixed_go<6, 1>(cuts, G);
        break;
    default:
        gram_mixed_go<3, 2>(cuts, G);
        gram_mixed_go<4, 2>(cuts, G);
        gram_mixed_go<5, 2>(cuts, G);
        gram_mixed_go<6, 2>(cuts, G);
    }
    return hipGetLastError();
}
