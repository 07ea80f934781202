// lekf_trf.hpp -- the local solve without eigenvalues, on a P x P grid of lanes (P = 8).
//
// The analysis needs three functions of A = C + (k-1)/alpha I (k x k, positive
// definite): A^-1 b and, for each state row x, x A^-1/2 and x A^-1 b.  With the
// Householder form A = Q T Q^T they are (x Q) f(T) Q^T, and f(T) z is a sum of
// tridiagonal solves, T^-1/2 z ~ sum_j om_j (T + sg_j I)^-1 z (lekf_invsqrt.hpp):
// all terms positive, 16 to 24 of them for the condition numbers of most local lists,
// to rounding.  Against tridiagonalisation + QL + rotation replay this drops Q
// (4k^3/3 flops and 2 k^2 values out and in), the scalar QL recurrence (one lane
// per point) and the rotation streams (46 KB written and read twice per point at
// k = 50); what is left is independent across shifts and rows.
//
// Layout: index i of a point belongs to grid coordinate i % P and slot i / P, so
// lane (r, c) of the grid holds elements (r + P a, c + P b) of A in registers
// M[a][b], and the trailing blocks of a Householder step stay spread over all
// lanes.  The rows to transform (X: the state rows, then b) hang below the matrix:
// row g on grid row g % P, slot g / P.  A step reads one row of M through LDS
// (which gives the reflector in both directions, M being symmetric), and all sums
// over grid rows or columns are DPP butterflies.  The reflectors stay in M's
// finished rows.  Sums run in an order that depends on the indices alone, and
// slots past k add exact zeros; products are fused into sums only where an fma is
// written (the compiler's own choice differs between numbers of slots, which come from
// the launch's largest k), so a point's bits do not depend on the launch.
#pragma once
#include "lekf_dev.hpp"
#include "lekf_invsqrt.hpp"

namespace {

__device__ constexpr lekf_invsqrt::Table g_invsqrt = lekf_invsqrt::make_table();

constexpr int P = 8;  // the wave's grid of lanes

// LDS stride of a vector stored [coordinate][slot]: even (16-byte reads) and such
// that the P coordinates' reads fall on distinct banks
__host__ __device__ constexpr int trf_ld(int NB) { return NB <= 10 ? 10 : 14; }

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double xor_f64(double x, int j, int lane)
{
    const long long b = __double_as_longlong(x);
    const int lo = lane_xor((int)b, j, lane), hi = lane_xor((int)(b >> 32), j, lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum over the P lanes of a grid row (c), in every lane
__device__ __forceinline__ double grid_sum_c(double x)
{
    x += dpp_f64<0xB1>(x);   // quad_perm [1,0,3,2]
    x += dpp_f64<0x4E>(x);   // quad_perm [2,3,0,1]
    x += dpp_f64<0x141>(x);  // row_half_mirror: the other quad
    return x;
}

// sum over the grid rows (r) of a value that is the same in every lane of a row
__device__ __forceinline__ double grid_sum_r(double x, int lane)
{
    x += dpp_f64<0x128>(x);  // row_ror:8
    x += xor_f64(x, 16, lane);
    x += xor_f64(x, 32, lane);
    return x;
}

// v[0..P-1] summed over the P lanes of a grid row, element c to lane c
__device__ __forceinline__ double grid_scatter_c(double (&v)[P], int c)
{
#pragma unroll
    for (int u = 0; u < P / 2; ++u) {
        const double keep = (c & 4) ? v[u + P / 2] : v[u], send = (c & 4) ? v[u] : v[u + P / 2];
        v[u] = keep + dpp_f64<0x141>(send);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const double keep = (c & 2) ? v[u + 2] : v[u], send = (c & 2) ? v[u] : v[u + 2];
        v[u] = keep + dpp_f64<0x4E>(send);
    }
    const double keep = (c & 1) ? v[1] : v[0], send = (c & 1) ? v[0] : v[1];
    return keep + dpp_f64<0xB1>(send);
}

// Householder steps s = P T .. P T + P - 1 of the point's matrix (those below
// k - 2), each applied to M from both sides and to the rows X from the right:
// H = I - tau v v^T, v zero up to s, v[s+1] = v0.  On exit row s of M holds v
// (columns above s), es[s] the off-diagonal and ts[s] tau.  vx, vw: P * trf_ld doubles of
// LDS each, es and ts P * NB.  bad: an entry of the reduction was not finite.
template <int T, int NB, int NE>
__device__ __forceinline__ void trf_stage(double (&M)[NB][NB], double (&X)[NE][NB], int k, int r,
                                          int c, int lane, double* vx, double* vw,
                                          double* es, double* ts, bool& bad)
{
#pragma clang fp contract(off)
    constexpr int LD = trf_ld(NB);
    constexpr int T1 = T + 1 < NB ? T + 1 : T;
#pragma unroll 1
    for (int u = 0; u < P; ++u) {
        const int s = P * T + u;
        if (s >= k - 2) break;
        if (r == u) {
#pragma unroll
            for (int b = T; b < NB; ++b) vx[c * LD + b] = M[T][b];
        }
        __syncthreads();
        double xr[NB], xc[NB];
#pragma unroll
        for (int a = T; a < NB; ++a) {
            xr[a] = vx[r * LD + a];
            xc[a] = vx[c * LD + a];
        }
        const double x0 = u < P - 1 ? vx[(u + 1) * LD + T] : vx[T1];
        xr[T] = r > u ? xr[T] : 0.0;
        xc[T] = c > u ? xc[T] : 0.0;
        double n2 = 0.0;
#pragma unroll
        for (int b = T; b < NB; ++b) n2 = fma(xc[b], xc[b], n2);
        n2 = grid_sum_c(n2);
        bad |= !(n2 <= 1.0e300);
        const bool live = n2 > 1.0e-280;
        const double n2s = live ? n2 : 1.0;
        const double nrm = n2s * rsq_nr(n2s);
        const double al = x0 >= 0.0 ? -nrm : nrm;
        const double v0 = x0 - al;
        const double tau = live ? rcp_nr(nrm * (nrm + fabs(x0))) : 0.0;
        if (r == 0 && c == 0) {
            es[s] = live ? al : x0;
            ts[s] = tau;
        }
        if (live) {
            // v[s+1] = v0 in the reflector and in M's row s
            xr[T] = r == u + 1 ? v0 : xr[T];
            xc[T] = c == u + 1 ? v0 : xc[T];
            M[T][T] = (r == u && c == u + 1) ? v0 : M[T][T];
            if (T + 1 < NB) {
                xr[T1] = (u == P - 1 && r == 0) ? v0 : xr[T1];
                xc[T1] = (u == P - 1 && c == 0) ? v0 : xc[T1];
                M[T][T1] = (u == P - 1 && r == u && c == 0) ? v0 : M[T][T1];
            }
        }
        double p[NB], px[NE];
#pragma unroll
        for (int a = T; a < NB; ++a) {
            double t = M[a][T] * xc[T];
#pragma unroll
            for (int b = T + 1; b < NB; ++b) t = fma(M[a][b], xc[b], t);
            p[a] = grid_sum_c(t);
        }
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            double t = X[e][T] * xc[T];
#pragma unroll
            for (int b = T + 1; b < NB; ++b) t = fma(X[e][b], xc[b], t);
            px[e] = tau * grid_sum_c(t);
        }
        double pv = p[T] * xr[T];
#pragma unroll
        for (int a = T + 1; a < NB; ++a) pv = fma(p[a], xr[a], pv);
        pv = grid_sum_r(pv, lane);
        const double g = 0.5 * tau * tau * pv;
        // w = tau p - g v, zero up to s
#pragma unroll
        for (int a = T; a < NB; ++a) p[a] = fma(tau, p[a], -g * xr[a]);
        p[T] = r > u ? p[T] : 0.0;
        if (c == 0) {
#pragma unroll
            for (int a = T; a < NB; ++a) vw[r * LD + a] = p[a];
        }
        __syncthreads();
        double wc[NB];
#pragma unroll
        for (int b = T; b < NB; ++b) wc[b] = vw[c * LD + b];
#pragma unroll
        for (int a = T; a < NB; ++a)
#pragma unroll
            for (int b = T; b < NB; ++b)
                M[a][b] = fma(-p[a], xc[b], fma(-xr[a], wc[b], M[a][b]));
#pragma unroll
        for (int e = 0; e < NE; ++e)
#pragma unroll
            for (int b = T; b < NB; ++b) X[e][b] = fma(-px[e], xc[b], X[e][b]);
    }
}

template <int T, int NB, int NE>
__device__ __forceinline__ void trf_reduce(double (&M)[NB][NB], double (&X)[NE][NB], int k, int r,
                                           int c, int lane, double* vx, double* vw,
                                           double* es, double* ts, bool& bad)
{
    trf_stage<T, NB, NE>(M, X, k, r, c, lane, vx, vw, es, ts, bad);
    if constexpr (T + 1 < NB)
        trf_reduce<T + 1, NB, NE>(M, X, k, r, c, lane, vx, vw, es, ts, bad);
}

// The diagonal to ds and the last off-diagonal to es (es[k-1] = 0).
template <int NB>
__device__ __forceinline__ void trf_diagonal(const double (&M)[NB][NB], int k, int r, int c,
                                             double* ds, double* es)
{
#pragma unroll
    for (int a = 0; a < NB; ++a)
        if (r == c && r + P * a < k) ds[r + P * a] = M[a][a];
    if (k >= 2) {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = a; b <= a + 1 && b < NB; ++b)
                if (r + P * a == k - 2 && c + P * b == k - 1) es[k - 2] = M[a][b];
    }
    if (r == 0 && c == 0) es[k - 1] = 0.0;
}

// Smallest table level whose interval [m, m kappa] reaches hi; kLevels if none
// does (or a bound is not a number).
__device__ __forceinline__ int trf_level(double hi, double m)
{
    double kap = 4.0;
    int l = 0;
    while (l < lekf_invsqrt::kLevels && !(hi <= m * kap)) {
        ++l;
        kap *= 8.0;
    }
    return l;
}

// f(T) of the rows of row group e (grid row r: row P e + r): the state rows get
// scale * T^-1/2, the row of b (grid row rb of this group, -1: none) T^-1.
// Lane (r, c) solves row r at shift c of each pass of P shifts; the P solutions are
// summed on the way back and element i = c + P b of the result lands in out[b] of
// lane c.  zrow: this lane's row in LDS; de: (d_i, e_i) pairs with (1, 0) from k on;
// tl: (P + 1) * ldt doubles for the factors e_i / delta_i of the P shifts (b's own
// shift 0 in the last).  The y of the forward pass stay in registers.
template <int NB>
__device__ __forceinline__ void trf_function(const double* zrow, const double2* de, int k, int lev,
                                             double m, double scale, int rb, int r, int c,
                                             double* tl, int ldt, double (&out)[NB])
{
#pragma clang fp contract(off)
#pragma unroll
    for (int b = 0; b < NB; ++b) out[b] = 0.0;
    const int N = 8 + 4 * lev;
    const bool isb = r == rb;
    // one grid row writes the factors of the shifts; b's lane of shift 0 its own
    const bool shared = r == (rb == 0 ? 1 : 0), own = isb && c == 0;
    double* tw = tl + (own ? P : c) * ldt;
    for (int pass = 0; pass * P < N; ++pass) {
        const int j = pass * P + c;
        double sh = m, wt = 0.0;
        if (own) {
            sh = 0.0;
            wt = pass == 0 ? 1.0 : 0.0;
        } else if (j < N) {
            sh = m * g_invsqrt.sg[lev][j];
            wt = isb ? 0.0 : scale * g_invsqrt.om[lev][j];
        }
        double y[P * NB];
        double t = 0.0, yp = 0.0, ep = 0.0;
#pragma unroll
        for (int i = 0; i < P * NB; ++i)
            if (i < k) {
                const double2 q = de[i];
                const double rr = rcp_nr(fma(-ep, t, q.x + sh));
                yp = fma(-t, yp, wt * zrow[i]);
                y[i] = yp * rr;
                t = q.y * rr;
                ep = q.y;
                if (shared || own) tw[i] = t;
            }
        __syncthreads();
        double x = 0.0;
#pragma unroll
        for (int b = NB - 1; b >= 0; --b)
            if (P * b < k) {
                double v[P];
#pragma unroll
                for (int u = P - 1; u >= 0; --u) {
                    const int i = P * b + u;
                    v[u] = 0.0;
                    if (i < k) {
                        x = fma(-tw[i], x, y[i]);
                        v[u] = x;
                    }
                }
                out[b] += grid_scatter_c(v, c);
            }
        __syncthreads();
    }
}

// rows <- rows H_s for s = P T + P - 1 down to P T (those below k - 2); vst: the
// stage's P reflectors in LDS, [u][coordinate][slot]; ts: tau
template <int T, int NB, int NE>
__device__ __forceinline__ void trf_back_stage(double (&out)[NE][NB], int k, int c,
                                               const double* vst, const double* ts)
{
#pragma clang fp contract(off)
    constexpr int LD = trf_ld(NB);
#pragma unroll 1
    for (int u = P - 1; u >= 0; --u) {
        const int s = P * T + u;
        if (s >= k - 2) continue;
        const double tau = ts[s];
        double v[NB];
#pragma unroll
        for (int b = T; b < NB; ++b) v[b] = vst[(u * P + c) * LD + b];
        v[T] = c > u ? v[T] : 0.0;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            double t = out[e][T] * v[T];
#pragma unroll
            for (int b = T + 1; b < NB; ++b) t = fma(out[e][b], v[b], t);
            t = tau * grid_sum_c(t);
#pragma unroll
            for (int b = T; b < NB; ++b) out[e][b] = fma(-t, v[b], out[e][b]);
        }
    }
}

}  // namespace
