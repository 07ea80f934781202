// lekf_trf.hip -- the plain local solve, 32 < k <= LEKF_KSPLIT (gfx950).
//
// Jobs that output neither trans nor pao take two kernels per sub-batch after the
// Gram, one wave per point each (lekf_trf.hpp): lekf_trd_kernel reduces
// C + (k-1)/alpha I to its tridiagonal T and carries the state rows and b through
// Q; lekf_trf_kernel evaluates the functions of T, carries the rows back and
// writes the analysis.  A point whose bounds put its condition number past the
// rational form's tables (or are not finite) is flagged, listed and left to
// lekf_eig_fix_kernel, whose Gram is still at the start of the record.
//
// Both are bound by VALU issue at two to four waves per SIMD (75% and 60% busy at k = 50;
// about 170 FP64 operations per Householder step, half of them the rank-2 update; a step's
// chain of reductions, rsq and rcp is what the second and third wave cover).
// Against the recorded-rotation solve it replaced for these jobs (Householder with Q,
// QL one lane per point, rotation replay), per cycle: radar 128 x 128 x 60, k = 50:
// 270 -> 43.5 ms (27.8 + 15.7); GFS-sized 192 x 94 x 64, k = 40: 171 -> 27 ms; 3001
// points at k = 80, where the matrix was in LDS: 24.9 -> 0.45 ms.
#include "lekf_ktime.hpp"
#include "lekf_split.hpp"
#include "lekf_trf.hpp"

namespace {

// grid slots (indices per lane and direction) of an ensemble size
__host__ __device__ constexpr int trf_slots(int k) { return (k + 7) / 8; }
__host__ __device__ constexpr int trf_ldz(int kmax) { return kmax | 1; }
__host__ __device__ constexpr int trd_lds_doubles(int NB, int nvmax, int kmax)
{
    return 16 * trf_ld(NB) + 24 * NB + LEKF_NVMAX + 1 + nvmax * trf_ldz(kmax);
}
__host__ __device__ constexpr int trf_lds_doubles(int NB, int NE, int kmax)
{
    // (d, e), tau, the row of b's solution, then rows and factors or a stage's reflectors
    const int a = (8 * NE + 9) * trf_ldz(8 * NB), b = 64 * trf_ld(NB);
    return 16 * NB + 8 * NB + 8 * NB + LEKF_NVMAX + 1 + 1 + (a > b ? a : b);
}

// The state rows of a point: row v of nrow (3-D rows, then at level 0 the 2-D ones)
struct PointRows {
    int n3, nrow, lev, ij;
};
__device__ __forceinline__ PointRows point_rows(const LekfJob& J, int b)
{
    PointRows R{0, 0, 0, 0};
    if (J.flags & LEKF_F_APPLY) {
        R.lev = b / J.nij;
        R.ij = b - R.lev * J.nij;
        R.n3 = J.nv3d;
        R.nrow = R.n3 + (R.lev == 0 ? J.nv2d : 0);
    }
    return R;
}
__device__ __forceinline__ long row_off(const LekfJob& J, const PointRows& R, int b, int v)
{
    return v < R.n3 ? ((long)b * R.n3 + v) * J.k : ((long)R.ij * J.nv2d + (v - R.n3)) * J.k;
}

// Smallest and largest eigenvalue of the tridiagonal (ds, es), inside [0, hi]: half
// the wave sections the interval for each by counting negative pivots.
__device__ void trf_extremes(const double* ds, const double* es, int k, int lane, double hi,
                             double& lmin, double& lmax)
{
    const bool top = lane < 32;
    const int l = lane & 31;
    double a[2] = {0.0, 0.0}, b[2] = {hi, hi};
    for (int it = 0; it < 8; ++it) {
        const double lo = top ? a[0] : a[1], w = (top ? b[0] : b[1]) - lo;
        const double x = lo + w * ((l + 1) * (1.0 / 33.0));
        int cnt = 0;
        double q = 1.0, e2 = 0.0;
        for (int i = 0; i < k; ++i) {
            q = ds[i] - x - (i ? e2 / q : 0.0);
            if (q == 0.0) q = -1.0e-300;
            cnt += q < 0.0;
            e2 = es[i] * es[i];
        }
        // above: the wanted eigenvalue lies above x
        const unsigned long long above = __ballot(top ? cnt < k : cnt == 0);
        const int na[2] = {(int)__popcll(above & 0xffffffffull), (int)__popcll(above >> 32)};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double l0 = a[h], wh = b[h] - l0;
            a[h] = l0 + wh * (na[h] * (1.0 / 33.0));
            b[h] = l0 + wh * ((na[h] + 1) * (1.0 / 33.0));
        }
    }
    lmax = 0.5 * (a[0] + b[0]);
    lmin = 0.5 * (a[1] + b[1]);
}

// Registers per lane: the matrix takes 2 NB^2 of them until its slots are finished.  Held to
// these waves lekf_trd_kernel spills at NB = 5, 8 and 9 (72, 64 and 244 bytes a lane with one
// row group, 164, 212 and 404 with three).  20,000 points, ms with one wave per SIMD fewer:
// one group k = 40 0.36 (0.34 so), k = 64 1.44 (0.91), k = 72 1.76 (1.50); three groups k = 40
// 0.42 (0.56), k = 64 1.53 (1.22), k = 72 1.92 (2.67): the two slower ones are the price of one
// rule for both.
constexpr int trd_waves_per_simd(int nb) { return nb <= 5 ? 4 : nb <= 6 ? 3 : nb <= 9 ? 2 : 1; }
constexpr int trf_waves_per_simd(int nb) { return nb <= 5 ? 4 : nb <= 7 ? 3 : nb <= 8 ? 2 : 1; }

// mode: the launch's Gram arithmetic (0 FP64); kthr, rlist, lcap: the mixed
// forms' redo list (see lekf_ql_kernel)
template <int NB, int NE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(trd_waves_per_simd(NB))))
void lekf_trd_kernel(const LekfJob* __restrict__ jobs, int njobs, long gp0,
                     double* __restrict__ ws, long gstride, int nvmax, int kmax, int pass,
                     int mode, double kthr, int* __restrict__ rlist, long lcap,
                     int* __restrict__ flist)
{
#pragma clang fp contract(off)
    extern __shared__ double smem[];
    constexpr int LD = trf_ld(NB);
    long gp;
    if (!split_slot_point(blockIdx.x, gp0, (long)gridDim.x, pass, rlist, gp)) return;
    const LekfJob& J = jobs[lekf_job_of(jobs, njobs, gp)];
    if (J.trans || J.pao) return;
    const int b = (int)(gp - J.pt_begin + J.pt0);
    const int p = J.loc_cnt ? J.loc_cnt[b] : (int)(J.loc_off[b + 1] - J.loc_off[b]);
    if (p <= 0) return;
    const int k = J.k, lane = threadIdx.x, r = lane >> 3, c = lane & 7;
    double* rec = ws + (long)blockIdx.x * gstride;
    const TrfRec S = trf_rec(kmax);
    double* vx = smem;
    double* vw = vx + P * LD;
    double* ds = vw + P * LD;
    double* es = ds + P * NB;
    double* ts = es + P * NB;
    double* mean = ts + P * NB;
    double* rows = mean + LEKF_NVMAX + 1;
    const int ldz = trf_ldz(kmax);

    double alpha = J.infl_in ? J.infl_in[b] : J.infl_fixed;
    if ((J.flags & LEKF_F_MINFL) && J.minfl > 0.0 && alpha < J.minfl) alpha = J.minfl;
    const double shift = (double)(k - 1) * (1.0 / alpha);
    const PointRows R = point_rows(J, b);
    for (int v = 0; v < R.nrow; ++v) {
        const double* src = (v < R.n3 ? J.x3b : J.x2b) + row_off(J, R, b, v);
        for (int i = lane; i < k; i += 64) rows[v * ldz + i] = src[i];
    }
    double M[NB][NB], X[NE][NB];
    double tr = 0.0;
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int i = r + P * a, j = c + P * q;
            M[a][q] = (i < k && j < k) ? rec[(long)i * k + j] : 0.0;
            if (a == q && i == j && i < k) {
                tr += M[a][q];
                M[a][q] += shift;
            }
        }
    __syncthreads();
    // the rows' means in member order (speedy/common/common_speedy.f90:335-370)
    if (lane < R.nrow) {
        const double* x = rows + lane * ldz;
        double s = x[0];
        for (int m = 1; m < k; ++m) s += x[m];
        mean[lane] = s / (double)k;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int g = P * e + r, i = c + P * q;
            double x = 0.0;
            if (i < k) {
                if (g < R.nrow)
                    x = rows[g * ldz + i] - mean[g];
                else if (g == nvmax)
                    x = rec[(long)k * k + i];
            }
            X[e][q] = x;
        }
    bool bad = false;
    trf_reduce<0, NB, NE>(M, X, k, r, c, lane, vx, vw, es, ts, bad);
    trf_diagonal<NB>(M, k, r, c, ds, es);
    __syncthreads();
    tr = wave_sum(tr);
    // bounds of the spectrum: C is positive semidefinite, so A >= shift up to the
    // Gram's rounding (1e-6 of its norm in the mixed forms); above, Gershgorin's
    // circles of T and the trace
    double hi = 0.0;
    for (int i = lane; i < k; i += 64) {
        const double h = fabs(ds[i]) + fabs(es[i]) + (i > 0 ? fabs(es[i - 1]) : 0.0);
        bad |= !(h <= 1.0e300);
        hi = h > hi ? h : hi;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double h = __shfl_xor(hi, o, 64);
        hi = h > hi ? h : hi;
    }
    const double htr = tr * (1.0 + 1.0e-5) + shift;
    hi = htr < hi ? htr : hi;
    bad = __ballot(bad) != 0ull;
    const double m = shift * (mode == 0 ? 0.999 : 0.75);
    const int lev = trf_level(hi, m);
    const bool hard = bad || lev >= (mode == 0 ? lekf_invsqrt::kLevels : 5);
    int redo = pass ? kSplitRedo : 0;
    if (!pass && kthr > 0.0 && !bad && J.hdxf && hi > kthr * 0.75 * shift) {
        double lmin, lmax;
        trf_extremes(ds, es, k, lane, hi, lmin, lmax);
        if (lmin > 0.0 && lmax > kthr * lmin) {
            int pos = 0;
            if (lane == 0) {
                pos = atomicAdd(rlist, 1);
                if (pos < lcap) rlist[1 + pos] = (int)gp;
            }
            pos = __builtin_amdgcn_readfirstlane(pos);
            if (pos < lcap) redo = kSplitRedo;
        }
    }
    if (lane == 0) {
        rec[gram_stride(kmax)] = (double)((hard ? kSplitOverflow : 0) | redo);
        rec[S.sc] = m;
        rec[S.sc + 1] = (double)lev;
        rec[S.sc + 2] = tr;
        if (hard && ((redo & kSplitRedo) != 0) == (pass != 0)) split_flag_slot(flist, blockIdx.x);
    }
    if (hard) return;
    for (int i = lane; i < k; i += 64) {
        rec[S.d + i] = ds[i];
        rec[S.e + i] = es[i];
        rec[S.tau + i] = i < k - 2 ? ts[i] : 0.0;
    }
    if (lane < R.nrow) rec[S.mean + lane] = mean[lane];
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int g = P * e + r, i = c + P * q;
            if (i < k && g <= nvmax) rec[S.z + (long)g * kmax + i] = X[e][q];
        }
    // reflector s: row s of M, columns above s
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int q = a; q < NB; ++q) {
            const int i = r + P * a, j = c + P * q;
            if (j < k && i < j) rec[S.v + (long)i * k + j] = M[a][q];
        }
}

// Back through Q, stage T and below: the stage's reflectors go to LDS while the
// next stage's are on their way.
template <int T, int NB, int NE>
__device__ __forceinline__ void trf_back(double (&out)[NE][NB], double (&st)[NB], int k, int r,
                                         int c, const double* V, double* vst, const double* ts)
{
    constexpr int LD = trf_ld(NB);
    __syncthreads();
#pragma unroll
    for (int q = T; q < NB; ++q) vst[(r * P + c) * LD + q] = st[q];
    __syncthreads();
    if constexpr (T > 0) {
        const int i = r + P * (T - 1);
#pragma unroll
        for (int q = T - 1; q < NB; ++q) {
            const int j = c + P * q;
            st[q] = (j < k && i < j) ? V[(long)i * k + j] : 0.0;
        }
    }
    trf_back_stage<T, NB, NE>(out, k, c, vst, ts);
    if constexpr (T > 0) trf_back<T - 1, NB, NE>(out, st, k, r, c, V, vst, ts);
}

template <int NB, int NE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(trf_waves_per_simd(NB))))
void lekf_trf_kernel(const LekfJob* __restrict__ jobs, int njobs, long gp0,
                     const double* __restrict__ ws, long gstride, int nvmax, int kmax, int pass,
                     const int* __restrict__ rlist)
{
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double smem[];
    constexpr int KP = P * NB, ldz = trf_ldz(KP);
    long gp;
    if (!split_slot_point(blockIdx.x, gp0, (long)gridDim.x, pass, rlist, gp)) return;
    const LekfJob& J = jobs[lekf_job_of(jobs, njobs, gp)];
    if (J.trans || J.pao) return;
    const int b = (int)(gp - J.pt_begin + J.pt0);
    const int p = J.loc_cnt ? J.loc_cnt[b] : (int)(J.loc_off[b + 1] - J.loc_off[b]);
    const double* rec = ws + (long)blockIdx.x * gstride;
    const int k = J.k, lane = threadIdx.x, r = lane >> 3, c = lane & 7;
    int flag = 0;
    if (p > 0) {
        flag = (int)rec[gram_stride(kmax)];
        if (((flag & kSplitRedo) != 0) != (pass != 0) || (flag & kSplitOverflow)) return;
    } else if (pass) {
        return;
    }
    const TrfRec S = trf_rec(kmax);
    double2* de = (double2*)smem;
    double* ts = smem + 2 * KP;
    double* yb = ts + KP;
    double* mean = yb + KP;
    double* zl = mean + LEKF_NVMAX + 2;
    double* tl = zl + 8 * NE * ldz;
    double alpha = J.infl_in ? J.infl_in[b] : J.infl_fixed;
    const PointRows R = point_rows(J, b);
    const uint32_t mask = J.upd_mask ? J.upd_mask[R.lev] : 0xffffffffu;

    if (p <= 0) {
        // no local obs (common_letkf.f90:82-96): T = sqrt(alpha) I
        for (int v = 0; v < R.nrow; ++v) {
            const double* src = (v < R.n3 ? J.x3b : J.x2b) + row_off(J, R, b, v);
            for (int i = lane; i < k; i += 64) zl[i] = src[i];
            __syncthreads();
            double s = zl[0];
            for (int i = 1; i < k; ++i) s += zl[i];
            const double mv = s / (double)k;
            const double sa = (v >= R.n3 || ((mask >> v) & 1u)) ? sqrt(alpha) : 1.0;
            double* dst = (v < R.n3 ? J.x3a : J.x2a) + row_off(J, R, b, v);
            for (int i = lane; i < k; i += 64) dst[i] = mv + sa * (zl[i] - mv);
            __syncthreads();
        }
        if (J.transm)
            for (int i = lane; i < k; i += 64) J.transm[(size_t)b * k + i] = 0.0;
        if (lane == 0) {
            if (J.infl_out) J.infl_out[b] = (J.flags & LEKF_F_FIXED_INFL) ? J.infl_fixed : alpha;
            if (J.status) J.status[b] = 0;
        }
        return;
    }

    for (int i = lane; i < KP; i += 64) {
        const bool in = i < k;
        de[i] = make_double2(in ? rec[S.d + i] : 1.0, in ? rec[S.e + i] : 0.0);
        ts[i] = in ? rec[S.tau + i] : 0.0;
    }
    for (int g = 0; g < 8 * NE; ++g)
        for (int i = lane; i < KP; i += 64)
            zl[g * ldz + i] = (i < k && g <= nvmax) ? rec[S.z + (long)g * kmax + i] : 0.0;
    if (lane < R.nrow) mean[lane] = rec[S.mean + lane];
    const double m = rec[S.sc];
    const int lev = (int)rec[S.sc + 1];
    const double scale = sqrt(m * (double)(k - 1));
    __syncthreads();
    double out[NE][NB];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const int rb = nvmax - P * e;  // grid row of b in this group
        trf_function<NB>(zl + (P * e + r) * ldz, de, k, lev, m, scale,
                            rb >= 0 && rb < P ? rb : -1, r, c, tl, ldz, out[e]);
        if (r == rb) {
#pragma unroll
            for (int q = 0; q < NB; ++q) yb[c + P * q] = out[e][q];
        }
    }
    // X' w-bar = (x Q) . (T^-1 Q^T b)
    __syncthreads();
    double cw[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NB; ++q) s = fma(zl[(P * e + r) * ldz + c + P * q], yb[c + P * q], s);
        cw[e] = grid_sum_c(s);
    }
    double st[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) st[q] = 0.0;
    {
        const int i = r + P * (NB - 1), j = c + P * (NB - 1);
        st[NB - 1] = (j < k && i < j) ? rec[S.v + (long)i * k + j] : 0.0;
    }
    trf_back<NB - 1, NB, NE>(out, st, k, r, c, rec + S.v, zl, ts);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const int g = P * e + r;
        if (g < R.nrow) {
            const bool upd = g >= R.n3 || ((mask >> g) & 1u);
            const long o = row_off(J, R, b, g);
            const double* src = (g < R.n3 ? J.x3b : J.x2b) + o;
            double* dst = (g < R.n3 ? J.x3a : J.x2a) + o;
            const double mv = mean[g];
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                const int i = c + P * q;
                if (i < k) dst[i] = upd ? mv + (cw[e] + out[e][q]) : mv + (src[i] - mv);
            }
        } else if (g == nvmax && J.transm) {
#pragma unroll
            for (int q = 0; q < NB; ++q) {
                const int i = c + P * q;
                if (i < k) J.transm[(size_t)b * k + i] = out[e][q];
            }
        }
    }
    if (lane == 0) {
        if ((J.flags & LEKF_F_MINFL) && J.minfl > 0.0 && alpha < J.minfl) alpha = J.minfl;
        if (J.infl_out)
            J.infl_out[b] = (J.flags & LEKF_F_FIXED_INFL)
                                ? J.infl_fixed
                                : adaptive_alpha(alpha, rec[(long)k * k + k],
                                                 rec[S.sc + 2] / (double)(k - 1),
                                                 rec[(long)k * k + k + 1]);
        // the condition number is below the tables' 2^26, so no eigenvalue is truncated
        if (J.status) J.status[b] = pass ? LEKF_PT_FP64 : 0;
    }
}

// the plain solve of a sub-batch: nvmax + 1 rows hang below the matrix, in one
// group of eight or three (up to 7 state rows, the models' 3-D fields; 8 to 16 pay for
// 24: 20,000 points at k = 50, reduction and functions 0.68 + 0.24 ms with 7 rows in
// all, 0.73 + 0.62 with 10, 0.76 + 0.66 with 16)
template <int NB, int NE>
static hipError_t launch_trf(long nb, hipStream_t st, const LekfJob* djobs, int njobs, long g0,
                             double* ws, long gs, int nvmax, int kmax, int pass, int mode,
                             double kthr, int* rlist, long lcap, int* flist)
{
    const size_t dlds = trd_lds_doubles(NB, nvmax, kmax) * sizeof(double);
    const size_t flds = trf_lds_doubles(NB, NE, kmax) * sizeof(double);
    {
        KTime kt(pass ? "redo_tri" : "eig_tri", st);
        hipLaunchKernelGGL((lekf_trd_kernel<NB, NE>), dim3((unsigned)nb), dim3(LEKF_WAVE), dlds, st,
                           djobs, njobs, g0, ws, gs, nvmax, kmax, pass, mode, kthr, rlist, lcap,
                           flist);
    }
    KTime kt(pass ? "redo_apply" : "eig_apply", st);
    hipLaunchKernelGGL((lekf_trf_kernel<NB, NE>), dim3((unsigned)nb), dim3(LEKF_WAVE), flds, st,
                       djobs, njobs, g0, ws, gs, nvmax, kmax, pass, rlist);
    return hipGetLastError();
}

}  // namespace

hipError_t lekf_trf_launch(long nb, hipStream_t st, const LekfJob* djobs, int njobs, long g0,
                           double* ws, long gs, int nvmax, int kmax, int pass, int mode,
                           double kthr, int* rlist, long lcap, int* flist)
{
    const bool one = nvmax + 1 <= 8;
    switch (trf_slots(kmax)) {
#define LEKF_TRF_CASE(NB)                                                                       \
    case NB:                                                                                    \
        return one ? launch_trf<NB, 1>(nb, st, djobs, njobs, g0, ws, gs, nvmax, kmax, pass,     \
                                       mode, kthr, rlist, lcap, flist)                          \
                   : launch_trf<NB, 3>(nb, st, djobs, njobs, g0, ws, gs, nvmax, kmax, pass,     \
                                       mode, kthr, rlist, lcap, flist);
        LEKF_TRF_CASE(5)
        LEKF_TRF_CASE(6)
        LEKF_TRF_CASE(7)
        LEKF_TRF_CASE(8)
        LEKF_TRF_CASE(9)
        LEKF_TRF_CASE(10)
        LEKF_TRF_CASE(11)
        LEKF_TRF_CASE(12)
#undef LEKF_TRF_CASE
    default: return hipErrorInvalidValue;
    }
}

