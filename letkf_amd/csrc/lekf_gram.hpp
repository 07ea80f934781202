// lekf_gram.hpp -- the Gram product of a point's local obs on MFMA.
#pragma once
#include "lekf_dev.hpp"

namespace {

// ---------------------------------------------------------------------------
// Gram products.  Lane l holds A[i = l%16][kk = l/16] and B[kk][j = l%16] of
// each 16x16x4 step (16x16x32 BF16: kk = 8*(l/16) .. +7).
//
// The local list is read in chunks of 64 entries: lane l loads entry q0 + l
// (obs index, weight rho/rdiag, departure) with one coalesced access, and the
// MFMA steps of the chunk take them from the owning lanes by shuffles.  All
// gathers of the chunk's Y rows are then independent loads, issued together,
// instead of one dependent index -> row chain per step.  Wave wv of nw takes
// every nw-th chunk.
// ---------------------------------------------------------------------------
// A point's obs: the list at its first entry, the obs table
struct GramIn {
    gptr<int> idx;
    gptr<double> rho, lrd, rdiag, dep, Y;  // lrd: rdiag per list entry, or null
    gptr<float> Yf;
    long y_so, y_sm;
    int p, k;
    bool wloc;
};
__device__ __forceinline__ GramIn gram_in(const LekfJob& J, long off, int p)
{
    GramIn I;
    I.idx = uniform_ptr(J.loc_idx + off);
    I.rho = uniform_ptr(J.loc_rho + off);
    I.lrd = uniform_ptr(J.loc_rdiag ? J.loc_rdiag + off : nullptr);
    I.rdiag = uniform_ptr(J.rdiag);
    I.dep = uniform_ptr(J.dep);
    I.Y = uniform_ptr(J.hdxf);
    I.Yf = uniform_ptr(J.hdxf32);
    I.y_so = (long)uniform64((unsigned long long)J.y_so);
    I.y_sm = (long)uniform64((unsigned long long)J.y_sm);
    I.p = __builtin_amdgcn_readfirstlane(p);
    I.k = __builtin_amdgcn_readfirstlane(J.k);
    I.wloc = __builtin_amdgcn_readfirstlane(J.flags & LEKF_F_WLOC) != 0;
    return I;
}

struct ObsChunk {
    int o;       // obs index (0 when past the end: a valid row, weighted 0)
    double w;    // rho / rdiag (1 / rdiag with rdiag_wloc), 0 past the end
    double d;    // departure
};

__device__ __forceinline__ ObsChunk stage_chunk(const GramIn& I, int q0, int lane, double& p3)
{
    ObsChunk c{0, 0.0, 0.0};
    const int q = q0 + lane;
    if (q < I.p) {
        c.o = I.idx[q];
        const double rho = I.rho[q];
        const double rd = I.lrd ? I.lrd[q] : I.rdiag[c.o];
        c.w = (I.wloc ? 1.0 : rho) / rd;
        c.d = I.dep[c.o];
        p3 += rho;
    }
    return c;
}

template <int NT>
__device__ __forceinline__ void gram_f64(const GramIn& I, int lane,
                                         lekf_d4* acc, double& p3, int wv, int nw)
{
    // k <= 32.  4-obs steps whose rows are gathered at once (bounded by the registers
    // the rows and the NT (NT + 1) / 2 accumulator tiles take)
    static_assert(NT <= 3, "whole tiles up to k = 32");
    constexpr int SUB = NT == 1 ? 16 : NT == 2 ? 8 : 4;
    const int lr = lane & 15, kq = lane >> 4, p = I.p, k = I.k;
    for (int q0 = 64 * wv; q0 < p; q0 += 64 * nw) {
        const ObsChunk ch = stage_chunk(I, q0, lane, p3);
#pragma unroll 1
        for (int h = 0; h < 16 && q0 + 4 * h < p; h += SUB) {
            double v[SUB][NT], wt[SUB];
#pragma unroll
            for (int st = 0; st < SUB; ++st) {
                const int src = 4 * (h + st) + kq;
                const int o = __shfl(ch.o, src, 64);
                const double w = __shfl(ch.w, src, 64);
                const double dd = __shfl(ch.d, src, 64);
                wt[st] = w;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int c = 16 * t + lr;
                    double x = 0.0;
                    if (c < k)
                        x = I.Y[(long)o * I.y_so + (long)c * I.y_sm];
                    else if (c == k)
                        x = dd;
                    v[st][t] = x;
                }
            }
#pragma unroll
            for (int st = 0; st < SUB; ++st) {
                int a = 0;
#pragma unroll
                for (int It = 0; It < NT; ++It) {
                    const double ai = wt[st] * v[st][It];
#pragma unroll
                    for (int Jt = It; Jt < NT; ++Jt) {
                        acc[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, v[st][Jt], acc[a], 0, 0, 0);
                        ++a;
                    }
                }
            }
        }
    }
}

// Mixed form: Y from the FP32 table, products accumulated in FP32 on MFMA.
// FP32: v_mfma_f32_16x16x4f32 (operands rounded to FP32).
// BF16x3: each FP32 operand split x = h + l (h = bf16(x), l = bf16(x - h));
// A*B ~ Ah*Bh + Ah*Bl + Al*Bh on v_mfma_f32_16x16x32_bf16.
// FP32 form: the FP32 accumulators are added into FP64 ones (accd) after each
// chunk of 64 obs, so no FP32 sum runs over more than 64 products and the
// rounding of long local lists (p ~ 10^3) does not build up.  The BF16x3 form
// keeps FP32 accumulation: its two-term split carries about 16 significant
// bits, which dominates its error, and the FP64 accumulators would cost it
// occupancy.
template <int NT>
__device__ __forceinline__ void mix_flush(lekf_f4* acc, lekf_d4* accd)
{
#pragma unroll
    for (int a = 0; a < NT * (NT + 1) / 2; ++a) {
#pragma unroll
        for (int r = 0; r < 4; ++r) accd[a][r] += (double)acc[a][r];
        acc[a] = lekf_f4{0.f, 0.f, 0.f, 0.f};
    }
}

template <int NT>
__device__ __forceinline__ void gram_f32(const GramIn& I, int lane,
                                         lekf_f4* acc, lekf_d4* accd, double& p3, int wv, int nw)
{
    constexpr int SUB = NT == 1 ? 16 : NT == 2 ? 8 : NT == 3 ? 4 : NT == 4 ? 2 : 1;
    const int lr = lane & 15, kq = lane >> 4, p = I.p, k = I.k;
    for (int q0 = 64 * wv; q0 < p; q0 += 64 * nw) {
        const ObsChunk ch = stage_chunk(I, q0, lane, p3);
        const float wf = (float)ch.w, df = (float)ch.d;  // one dword each across lanes
#pragma unroll 1
        for (int h = 0; h < 16 && q0 + 4 * h < p; h += SUB) {
            float v[SUB][NT], wt[SUB];
#pragma unroll
            for (int st = 0; st < SUB; ++st) {
                const int src = 4 * (h + st) + kq;
                const int o = __shfl(ch.o, src, 64);
                const float w = __shfl(wf, src, 64);
                const float dd = __shfl(df, src, 64);
                wt[st] = w;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int c = 16 * t + lr;
                    float x = 0.0f;
                    if (c < k)
                        x = I.Yf[(long)o * k + c];
                    else if (c == k)
                        x = dd;
                    v[st][t] = x;
                }
            }
#pragma unroll
            for (int st = 0; st < SUB; ++st) {
                int a = 0;
#pragma unroll
                for (int It = 0; It < NT; ++It) {
                    const float ai = wt[st] * v[st][It];
#pragma unroll
                    for (int Jt = It; Jt < NT; ++Jt) {
                        acc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai, v[st][Jt], acc[a], 0, 0, 0);
                        ++a;
                    }
                }
            }
        }
        mix_flush<NT>(acc, accd);
    }
}

// Split-BF16x3: K = 32 obs per MFMA step, two steps per chunk.  Lane l
// supplies 8 consecutive k values (kk = 8*(l/16) .. +7) of row/col l%16.
template <int NT>
__device__ __forceinline__ void gram_bf16x3(const GramIn& I, int lane,
                                            lekf_f4* acc, double& p3, int wv, int nw)
{
    const int lr = lane & 15, kq = lane >> 4, p = I.p, k = I.k;
    for (int q0 = 64 * wv; q0 < p; q0 += 64 * nw) {
        const ObsChunk ch = stage_chunk(I, q0, lane, p3);
        // the weight and departure in the precision the products use, so each
        // crosses lanes as one dword
        const float wf = (float)ch.w, df = (float)ch.d;
        for (int h = 0; h < 64 && q0 + h < p; h += 32) {
            lekf_bf8 ah[NT], al[NT], bh[NT], bl[NT];
            float wv8[8], dv8[8];
            int ov[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int src = h + 8 * kq + e;
                ov[e] = __shfl(ch.o, src, 64);
                wv8[e] = __shfl(wf, src, 64);
                dv8[e] = __shfl(df, src, 64);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int c = 16 * t + lr;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = 0.0f;
                    if (c < k)
                        x[e] = I.Yf[(long)ov[e] * k + c];
                    else if (c == k)
                        x[e] = dv8[e];
                }
                // two elements per rounding instruction (round to nearest even,
                // as the scalar conversion does)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const lekf_f2v xv = {x[e], x[e + 1]};
                    const lekf_f2v xa = {wv8[e] * x[e], wv8[e + 1] * x[e + 1]};
                    const lekf_b2v hb = __builtin_convertvector(xv, lekf_b2v);
                    const lekf_b2v ha = __builtin_convertvector(xa, lekf_b2v);
                    const lekf_f2v rb = {x[e] - (float)hb.x, x[e + 1] - (float)hb.y};
                    const lekf_f2v ra = {xa.x - (float)ha.x, xa.y - (float)ha.y};
                    const lekf_b2v lb = __builtin_convertvector(rb, lekf_b2v);
                    const lekf_b2v la = __builtin_convertvector(ra, lekf_b2v);
                    bh[t][e] = hb.x;
                    bh[t][e + 1] = hb.y;
                    bl[t][e] = lb.x;
                    bl[t][e + 1] = lb.y;
                    ah[t][e] = ha.x;
                    ah[t][e + 1] = ha.y;
                    al[t][e] = la.x;
                    al[t][e + 1] = la.y;
                }
            }
            int a = 0;
#pragma unroll
            for (int It = 0; It < NT; ++It) {
#pragma unroll
                for (int Jt = It; Jt < NT; ++Jt) {
                    acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[It], bh[Jt], acc[a], 0, 0, 0);
                    acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[It], bl[Jt], acc[a], 0, 0, 0);
                    acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[It], bh[Jt], acc[a], 0, 0, 0);
                    ++a;
                }
            }
        }
    }
}

// Write the upper tiles of G into LDS: C (k x k at A, leading dimension lda,
// exactly symmetric), b and sum w d^2; with add, accumulate onto what an
// earlier wave stored.  Only (row <= col) elements are taken so C is
// symmetric bit for bit.  Result-tile layouts (measured on gfx950): the FP64
// 16x16x4 MFMA puts element (row = l/16 + 4r, col = l%16) in register r of
// lane l; the FP32 and BF16 16x16 forms put (row = 4*(l/16) + r, col = l%16)
// there.
template <int NT, bool F64, typename ACC>
__device__ __forceinline__ void store_gram(const ACC* acc, int k, int lda, int lane, double* A,
                                           double* B, double* sumwd2, bool add)
{
    const int lr = lane & 15, kq = lane >> 4;
    int a = 0;
#pragma unroll
    for (int I = 0; I < NT; ++I) {
#pragma unroll
        for (int Jt = I; Jt < NT; ++Jt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * I + (F64 ? kq + 4 * r : 4 * kq + r);
                const int col = 16 * Jt + lr;
                const double val = (double)acc[a][r];
                if (row <= col) {
                    if (col < k) {
                        const double v = add ? A[row * lda + col] + val : val;
                        A[row * lda + col] = v;
                        A[col * lda + row] = v;
                    } else if (col == k) {
                        if (row < k)
                            B[row] = add ? B[row] + val : val;
                        else
                            *sumwd2 = add ? *sumwd2 + val : val;
                    }
                }
            }
            ++a;
        }
    }
}

// FP64 Gram of k > 32 with the columns cut to fit: NTF full 16-column tiles, then NS
// strips of 4 columns (16 NTF + 4 NS >= k + 1, columns k..: the departure, zeros).
// Full tiles go through v_mfma_f64_16x16x4f64; a strip against a tile, or against
// another strip, is one v_mfma_f64_4x4x4f64, whose four blocks take the tile's 16
// rows as they lie and the strip's 4 columns repeated.  At the nominal 64 and 16 cycles
// that is 448 instead of 640 cycles per 4 obs at k = 50 (k + 1 rounded up to 52 instead
// of 64).  From 9 columns in the last tile on the strips would take as long as the tile;
// strips alone, without tiles, are no faster (151-155 ms where this takes 147) since they
// need the rows turned by vector instructions.  4x4x4 lanes
// (measured): A[i][kk] of block q in lane 16 kk + 4 q + i, B[kk][j] in
// 16 kk + 4 q + j, D[i][j] in 16 i + 4 q + j.
//
// The rows of one pair of 4-obs steps are loaded while the previous pair's products
// run.  ROWS: Y(o, m) = hdxf[o * y_so + m] with 0 <= y_so < 2^29 (an obs's row costs
// one multiply-add and the columns are immediate offsets), else any strides.
__host__ __device__ constexpr int gram_ntf(int k) { return (k + 1 + 7) / 16; }
__host__ __device__ constexpr int gram_ns(int k)
{
    const int r = k + 1 - 16 * gram_ntf(k);
    return r <= 0 ? 0 : (r + 3) / 4;
}

// the cuts of 32 < k <= 95, numbered
constexpr int kGramCuts = 13;
__host__ __device__ constexpr int gram_cut(int ntf, int ns) { return 3 * (ntf - 2) + ns; }

template <int NTF, int NS>
struct GramAcc {
    static constexpr int NT = NTF * (NTF + 1) / 2;
    lekf_d4 t[NT];
    double s[NTF * NS + NS * (NS + 1) / 2 + 1];  // tile rows x strips, then strip pairs
};

// Where a lane reads its columns of a row: the tile columns from lr on, then the columns
// of the strips (NS = 0: of the last tile), those past the end as the row's first
template <int NTF, int NS>
struct RowLane {
    static constexpr int NF = NS > 0 ? NTF : NTF - 1;  // tiles with every column below k
    static constexpr int NX = NS > 0 ? NS : 1;
    gptr<double> base;  // Y and the lane's first column
    long off[NX];       // elements from base
    bool in[NX];        // column below k (else the departure, column k, or unused)
};
template <int NTF, int NS, bool ROWS>
__device__ __forceinline__ RowLane<NTF, NS> row_lane(const GramIn& I, int lane)
{
    RowLane<NTF, NS> R;
    const int lr = lane & 15;
    const long sm = ROWS ? 1 : I.y_sm;
    R.base = I.Y + lr * sm;
#pragma unroll
    for (int x = 0; x < R.NX; ++x) {
        const int c = NS > 0 ? 16 * NTF + 4 * x + (lr & 3) : 16 * (NTF - 1) + lr;
        R.in[x] = c < I.k;
        R.off[x] = ((c < I.k ? c : 0) - lr) * sm;
    }
    return R;
}

template <int NTF, int NS, bool ROWS>
__device__ __forceinline__ void gram_rows(const GramIn& I, const RowLane<NTF, NS>& R,
                                          const ObsChunk& ch, int h, int kq,
                                          double (&v)[2][NTF + NS], double (&wt)[2],
                                          double (&dd)[2])
{
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        const int src = 4 * (h + st) + kq;
        const int o = __shfl(ch.o, src, 64);
        wt[st] = __shfl(ch.w, src, 64);
        dd[st] = __shfl(ch.d, src, 64);
        gptr<double> row;
        if (ROWS)  // one multiply-add: o * (8 y_so) + base, both factors below 2^32
            row = (gptr<double>)((unsigned long long)(unsigned)o * (unsigned)(8 * (unsigned)I.y_so) +
                                 (unsigned long long)R.base);
        else
            row = R.base + (long)o * I.y_so;
#pragma unroll
        for (int t = 0; t < R.NF; ++t) v[st][t] = ROWS ? row[16 * t] : row[16L * t * I.y_sm];
#pragma unroll
        for (int x = 0; x < R.NX; ++x) v[st][R.NF + x] = row[R.off[x]];
    }
}

template <int NTF, int NS>
__device__ __forceinline__ void gram_step(GramAcc<NTF, NS>& G, const RowLane<NTF, NS>& R,
                                          double (&v)[NTF + NS], double wt, double dd)
{
    // (the departure goes in here, not where the row is loaded: there it would wait for
    // the load before the previous pair's products)
#pragma unroll
    for (int x = 0; x < R.NX; ++x) v[R.NF + x] = R.in[x] ? v[R.NF + x] : dd;
    double a[NTF + NS];
#pragma unroll
    for (int t = 0; t < NTF + NS; ++t) a[t] = wt * v[t];
    int q = 0;
#pragma unroll
    for (int I = 0; I < NTF; ++I)
#pragma unroll
        for (int Jt = I; Jt < NTF; ++Jt, ++q)
            G.t[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[I], v[Jt], G.t[q], 0, 0, 0);
    q = 0;
#pragma unroll
    for (int I = 0; I < NTF + NS; ++I)
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (I < NTF || I - NTF <= s) {
                G.s[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[I], v[NTF + s], G.s[q], 0, 0, 0);
                ++q;
            }
}

template <int NTF, int NS, bool ROWS>
__device__ __forceinline__ void gram_strips(const GramIn& I, int lane, GramAcc<NTF, NS>& G,
                                            double& p3, int wv, int nw)
{
    const int kq = lane >> 4, p = I.p;
    const RowLane<NTF, NS> R = row_lane<NTF, NS, ROWS>(I, lane);
    for (int q0 = 64 * wv; q0 < p; q0 += 64 * nw) {
        const ObsChunk ch = stage_chunk(I, q0, lane, p3);
        const int n = p - q0 < 64 ? (p - q0 + 3) / 4 : 16;  // 4-obs steps (a pair's second
                                                            // may be past the end: weight 0)
        double va[2][NTF + NS], wa[2], da[2], vb[2][NTF + NS], wb[2], db[2];
        gram_rows<NTF, NS, ROWS>(I, R, ch, 0, kq, va, wa, da);
#pragma unroll 1
        for (int h = 0; h < n; h += 4) {
            if (h + 2 < n) gram_rows<NTF, NS, ROWS>(I, R, ch, h + 2, kq, vb, wb, db);
            gram_step<NTF, NS>(G, R, va[0], wa[0], da[0]);
            if (h + 1 < n) gram_step<NTF, NS>(G, R, va[1], wa[1], da[1]);
            if (h + 2 >= n) break;
            if (h + 4 < n) gram_rows<NTF, NS, ROWS>(I, R, ch, h + 4, kq, va, wa, da);
            gram_step<NTF, NS>(G, R, vb[0], wb[0], db[0]);
            if (h + 3 < n) gram_step<NTF, NS>(G, R, vb[1], wb[1], db[1]);
        }
    }
}

// The strip form's share of store_gram: C, b and sum w d^2 at A, B and sumwd2
template <int NTF, int NS>
__device__ __forceinline__ void store_strips(const GramAcc<NTF, NS>& G, int k, int lda, int lane,
                                             double* A, double* B, double* sumwd2, bool add)
{
    store_gram<NTF, true>(G.t, k, lda, lane, A, B, sumwd2, add);
    const int i = lane >> 4, q4 = (lane >> 2) & 3, j = lane & 3;
    int q = 0;
#pragma unroll
    for (int I = 0; I < NTF + NS; ++I)
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (I < NTF || I - NTF <= s) {
                const int row = I < NTF ? 16 * I + 4 * q4 + i : 16 * NTF + 4 * (I - NTF) + i;
                const int col = 16 * NTF + 4 * s + j;
                const double val = G.s[q];
                ++q;
                // a strip pair's four blocks are alike: block 0 writes it
                if (row <= col && (I < NTF || q4 == 0)) {
                    if (col < k) {
                        const double x = add ? A[row * lda + col] + val : val;
                        A[row * lda + col] = x;
                        A[col * lda + row] = x;
                    } else if (col == k) {
                        if (row < k)
                            B[row] = add ? B[row] + val : val;
                        else
                            *sumwd2 = add ? *sumwd2 + val : val;
                    }
                }
            }
}

}  // namespace

// the Gram of nb slots into the workspace records (lekf_gram.hip), one launch per form
// that the jobs' sizes take (outs: their cuts)
hipError_t lekf_gram_launch(int mode, int W, int kmax, int outs, long nb, hipStream_t st,
                            const LekfJob* djobs, int njobs, long g0, double* ws, long gs,
                            const int* rlist, int* zlist, int* flist);
