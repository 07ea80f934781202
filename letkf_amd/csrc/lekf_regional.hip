// lekf_regional.hip -- regional (SCALE-style) obs index and capped selection (gfx950).
//
// Obs index (scale/letkf/letkf_obs.f90:740-830, one subdomain): obs go to
// cell (ceiling(ri-0.5), ceiling(rj-0.5)) clamped to the grid, keeping input
// order within a cell (stable sort of unique keys cell << 32 | index).
//
// Selection (scale/letkf/letkf_tools.f90:853-1178): the rectangle of cells
// floor(ri -/+ dlon_zero) .. ceiling(...) is scanned row by row; a candidate
// passes when ndist = (sqrt(rdx^2+rdy^2)/sigma_h)^2 + (|dz|/sigma_v)^2 is not
// above the literal 13.33333333, with rloc = exp(-ndist/2) and
// rdiag = err^2/rloc.  Without a cap the accepted obs are emitted in scan
// order.
//
// The cap MAX_NOBS_PER_GRID = nobs_max > 0 (:1041-1156).  Per bucket (the
// reference's (element, obs type) pair) the reference keeps an
// insertion-sorted set of at most nobs_max obs by rdiag in storage slots: an
// obs that arrives while the set is not full takes the next free slot; later,
// an obs with rdiag strictly below the set's last-priority entry evicts that
// entry and takes over its slot (so an earlier obs wins a tie).  The kept obs
// are emitted bucket by bucket in slot order.  cap_slots gives the same slots
// without inserting serially:
//   * a candidate enters when fewer than nobs_max candidates before it in scan
//     order precede it in (rdiag, scan position) order, and the set after any
//     prefix is the nobs_max first entries of that prefix in this order;
//   * the set's last entry only moves down, so entries are evicted from the
//     largest down: the i-th candidate that enters a full set evicts the i-th
//     largest of the entries ever evicted, and takes its slot.
// A block of 256 candidates at a time is merged into the set held in LDS
// (ascending, double-buffered): each candidate's count of preceding entries
// is a binary search in the set plus a count over the block's earlier
// candidates, the new set and the block's evictions come from ranks in the
// union, and a candidate evicted within its own block passes its slot on
// (pointer jumping).
#include <algorithm>
#include <cmath>

#include "lekf_dev.hpp"
#include "lekf_regional.hpp"
#include "lekf_tune.hpp"
#include "lekf_ktime.hpp"

// Every FP64 operation in this file is rounded as written: no FMA contraction
// (the reference's results are reproduced operation by operation).
#pragma clang fp contract(off)

namespace {

constexpr double kNdMax = 13.33333333;  // scale/letkf/letkf_obs.f90:30

__device__ __forceinline__ unsigned long long lane_lt(int lane)
{
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

constexpr int kSelT = 256;  // threads per workgroup of the selection (4 waves)
constexpr int kSelW = kSelT / 64;

constexpr int kCapU = 1;               // candidates per thread in a block of the cap
constexpr int kCapB = kSelT * kCapU;   // candidates per block

// One block's potential entrants, entrants and evictions of the workgroup
// form of the cap (caps above LEKF_CAP_LDS, the kept set S in global memory).
struct CapLds {
    unsigned long long pkey[kCapB];  // potential entrants, scan order
    int ppos[kCapB];
    unsigned long long nkey[kCapB];  // entrants, scan order
    int npos[kCapB];
    int nc1[kCapB];                  // entries of S before each entrant
    int nU[kCapB];                   // entrant's rank in S + entrants
    unsigned long long ekey[kCapB];  // entrants, ascending
    int epos[kCapB];
    int ev[kCapB];                   // evictions, ascending: slot (>= 0) or -(entrant + 1)
    int slotn[kCapB];
    int link[kCapB];
    int wc[2][kCapU][kSelW];
};

// S in global memory (caps above LEKF_CAP_LDS): 2 * cap entries per array
struct CapGlobal {
    unsigned long long* key;
    int* pos;
    int* slot;
};

struct SelLds {
    CapLds cap;
    int seg_beg[LEKF_REG_SEG];
    int seg_pre[LEKF_REG_SEG + 1];
    int wcnt[kSelW][LEKF_REG_NB];
};

struct Cand {
    bool ok;
    int o, b;
    double rho, rd;
    unsigned long long bits;
};

struct ObsRec {
    double ri, rj, z, err;
    int b;
};

__device__ __forceinline__ ObsRec load_obs(const RegionalArgs& A, int o)
{
    ObsRec r;
    r.ri = A.ori[o];
    r.rj = A.orj[o];
    r.z = A.oz[o];
    r.err = A.oerr[o];
    r.b = A.obkt[o];
    return r;
}

// The reference's test and weights (scale/letkf/letkf_tools.f90:978-1037),
// each operation rounded as written (no contraction), so the cutoff decision
// and rdiag are bit-identical to the reference's.
__device__ __forceinline__ Cand eval_rec(const RegionalArgs& A, const ObsRec& r, int o, double ri,
                                         double rj, double rz)
{
    Cand c;
    const double rdx = rn_mul(rn_sub(ri, r.ri), A.dx);
    const double rdy = rn_mul(rn_sub(rj, r.rj), A.dy);
    const double nd_h = rn_div(__dsqrt_rn(rn_add(rn_mul(rdx, rdx), rn_mul(rdy, rdy))),
                                  A.sigma_h);
    const double nd_v = rn_div(fabs(rn_sub(r.z, rz)), A.sigma_v);
    const double nd = rn_add(rn_mul(nd_h, nd_h), rn_mul(nd_v, nd_v));
    c.o = o;
    c.ok = !(nd > kNdMax);
    c.b = r.b;
    c.rho = 0.0;
    c.rd = 0.0;
    c.bits = 0;
    if (c.ok) {
        c.rho = exp(-0.5 * nd);
        c.rd = rn_div(rn_mul(r.err, r.err), c.rho);
        c.bits = (unsigned long long)__double_as_longlong(c.rd);
    }
    return c;
}

// candidate q of the point's scan (row segments in LDS)
__device__ __forceinline__ int cand_obs(const SelLds& S, int nseg, int q, int& seg)
{
    while (seg + 1 < nseg && S.seg_pre[seg + 1] <= q) ++seg;
    return S.seg_beg[seg] + (q - S.seg_pre[seg]);
}

// Block-wide compaction of U flags per thread in (u, thread) order: pos[u]
// is the position of entry u among the flagged ones, tot their number.  The
// counts alternate between two buffers, so one barrier suffices.  Uniform
// call.
template <int U>
__device__ __forceinline__ void block_rank(int (*wc)[U][kSelW], int& par, const bool (&flag)[U],
                                           int tid, int (&pos)[U], int& tot)
{
    const int lane = tid & 63, wv = tid >> 6;
    unsigned long long m[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        m[u] = __ballot(flag[u]);
        if (lane == 0) wc[par][u][wv] = __popcll(m[u]);
    }
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int off = 0, t = 0;
#pragma unroll
        for (int w = 0; w < kSelW; ++w) {
            const int c = wc[par][u][w];
            off += w < wv ? c : 0;
            t += c;
        }
        pos[u] = base + off + __popcll(m[u] & lane_lt(lane));
        base += t;
    }
    tot = base;
    par ^= 1;
}

// V binary searches in lockstep (their loads overlap): out[v] = entries of the
// ascending (key, candidate) array [0, n) before (x[v], xp[v])
template <int V>
__device__ __forceinline__ void count_before(const unsigned long long* key, const int* pos, int n,
                                             const unsigned long long (&x)[V],
                                             const int (&xp)[V], int (&out)[V])
{
    int lo[V], hi[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        lo[v] = 0;
        hi[v] = n;
    }
    for (int w = n; w > 0; w >>= 1) {
        unsigned long long y[V];
        int yp[V], mid[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            mid[v] = (lo[v] + hi[v]) >> 1;
            const int m = mid[v] < n ? mid[v] : 0;
            y[v] = key[m];
            yp[v] = pos[m];
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (lo[v] < hi[v]) {
                if (y[v] < x[v] || (y[v] == x[v] && yp[v] < xp[v]))
                    lo[v] = mid[v] + 1;
                else
                    hi[v] = mid[v];
            }
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) out[v] = lo[v];
}

// The reference's cap (scale/letkf/letkf_tools.f90:1041-1156) over one
// bucket's candidates 0..n-1 in scan order, keyat(i) the priority key of
// candidate i (smaller first), by all kSelT threads of a workgroup with the
// kept set in global memory (caps above LEKF_CAP_LDS).  Returns the kept
// count; the kept entries are G[buf][0..kept) with pos = candidate and
// slot = storage slot (the output position).  Uniform call.
template <class KeyAt>
__device__ int cap_slots(CapLds& L, const CapGlobal& G, KeyAt keyat, int n, int cap, int tid,
                         int& bufo)
{
    constexpr bool kLds = false;
    constexpr int U = kCapU;
    constexpr int V = LEKF_CAP_LDS / kSelT;  // S entries per thread per round of the merge
    int s = 0, buf = 0, par = 0;
    unsigned long long xn[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = u * kSelT + tid;
        xn[u] = i < n ? keyat(i) : 0ull;
    }
    for (int b0 = 0; b0 < n; b0 += kCapB) {
        (void)kLds;
        unsigned long long* Sk = G.key + (size_t)buf * cap;
        int* Sp = G.pos + (size_t)buf * cap;
        int* Ss = G.slot + (size_t)buf * cap;
        unsigned long long* Tk = G.key + (size_t)(buf ^ 1) * cap;
        int* Tp = G.pos + (size_t)(buf ^ 1) * cap;
        int* Ts = G.slot + (size_t)(buf ^ 1) * cap;
        unsigned long long x[U];
        bool pot[U];
        const unsigned long long tau = s == cap ? Sk[cap - 1] : 0ull;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            x[u] = xn[u];
            const int i = b0 + u * kSelT + tid;
            // into a full set only below its last entry (a later candidate
            // with an equal key comes after it)
            pot[u] = i < n && (s < cap || x[u] < tau);
            const int inext = i + kCapB;  // the next block's keys, loaded ahead
            xn[u] = inext < n ? keyat(inext) : 0ull;
        }
        int pr[U], np;
        block_rank<U>(L.wc, par, pot, tid, pr, np);
        if (np == 0) continue;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (pot[u]) {
                L.pkey[pr[u]] = x[u];
                L.ppos[pr[u]] = b0 + u * kSelT + tid;
            }
        __syncthreads();
        // potential q = u * kSelT + tid of this thread: its entries of S
        // before it (c1) and the earlier potentials not above it (c2)
        unsigned long long y[U];
        int yp[U], c1[U], c2[U];
        int jmax = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = u * kSelT + tid;
            y[u] = q < np ? L.pkey[q] : ~0ull;
            yp[u] = q < np ? L.ppos[q] : 0;
            c2[u] = 0;
            if (q < np) jmax = q;
        }
        count_before<U>(Sk, Sp, s, y, yp, c1);
        {
            int j = 0;
            for (; j + 4 <= jmax; j += 4) {
                const unsigned long long k0 = L.pkey[j], k1 = L.pkey[j + 1];
                const unsigned long long k2 = L.pkey[j + 2], k3 = L.pkey[j + 3];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int q = u * kSelT + tid;
                    c2[u] += (j < q && k0 <= y[u]) + (j + 1 < q && k1 <= y[u]) +
                             (j + 2 < q && k2 <= y[u]) + (j + 3 < q && k3 <= y[u]);
                }
            }
            for (; j < jmax; ++j) {
                const unsigned long long k0 = L.pkey[j];
#pragma unroll
                for (int u = 0; u < U; ++u) c2[u] += (j < u * kSelT + tid && k0 <= y[u]);
            }
        }
        bool ent[U];
#pragma unroll
        for (int u = 0; u < U; ++u) ent[u] = u * kSelT + tid < np && c1[u] + c2[u] < cap;
        int er[U], e;
        block_rank<U>(L.wc, par, ent, tid, er, e);
        if (e == 0) continue;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (ent[u]) {
                L.nkey[er[u]] = y[u];
                L.npos[er[u]] = yp[u];
                L.nc1[er[u]] = c1[u];
            }
        __syncthreads();
        // entrant t = u * kSelT + tid: its rank among the entrants
        {
            unsigned long long xk[U];
            int r[U];
            int tmax = -1;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = u * kSelT + tid;
                xk[u] = t < e ? L.nkey[t] : 0ull;
                r[u] = 0;
                if (t < e) tmax = t;
            }
            if (tmax >= 0) {
                int w = 0;
                for (; w + 4 <= e; w += 4) {
                    const unsigned long long z0 = L.nkey[w], z1 = L.nkey[w + 1];
                    const unsigned long long z2 = L.nkey[w + 2], z3 = L.nkey[w + 3];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int t = u * kSelT + tid;
                        r[u] += (z0 < xk[u] || (z0 == xk[u] && w < t)) +
                                (z1 < xk[u] || (z1 == xk[u] && w + 1 < t)) +
                                (z2 < xk[u] || (z2 == xk[u] && w + 2 < t)) +
                                (z3 < xk[u] || (z3 == xk[u] && w + 3 < t));
                    }
                }
                for (; w < e; ++w) {
                    const unsigned long long z0 = L.nkey[w];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        r[u] += (z0 < xk[u] || (z0 == xk[u] && w < u * kSelT + tid));
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = u * kSelT + tid;
                if (t < e) {
                    L.ekey[r[u]] = xk[u];
                    L.epos[r[u]] = L.npos[t];
                    L.nU[t] = L.nc1[t] + r[u];
                }
            }
        }
        __syncthreads();
        const int snew = s + e < cap ? s + e : cap;
        const int nev = s + e - snew;
        // S entries move up by the entrants before them; the top nev leave
        for (int r0 = 0; r0 < s; r0 += V * kSelT) {
            unsigned long long xk[V];
            int xp[V], U2[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int r = r0 + v * kSelT + tid;
                xk[v] = r < s ? Sk[r] : ~0ull;
                xp[v] = r < s ? Sp[r] : 0x7fffffff;
            }
            count_before<V>(L.ekey, L.epos, e, xk, xp, U2);
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int r = r0 + v * kSelT + tid;
                if (r < s) {
                    const int Ur = r + U2[v];
                    if (Ur < cap) {
                        Tk[Ur] = xk[v];
                        Tp[Ur] = xp[v];
                        Ts[Ur] = Ss[r];
                    } else {
                        L.ev[Ur - cap] = Ss[r];
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = u * kSelT + tid;
            if (t < e) {
                const int Ut = L.nU[t];
                if (Ut < cap) {
                    Tk[Ut] = L.nkey[t];
                    Tp[Ut] = L.npos[t];
                } else {
                    L.ev[Ut - cap] = -(t + 1);
                }
            }
        }
        __syncthreads();
        // slots: the next free one while the set fills, then the slot of the
        // evicted entry, evictions taken from the largest down
        const int nfill = cap - s;
        bool chain = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = u * kSelT + tid;
            if (t < e) {
                int sl = -1, ln = -1;
                if (t < nfill) {
                    sl = s + t;
                } else {
                    const int v = L.ev[nev - 1 - (t - nfill)];
                    if (v >= 0)
                        sl = v;
                    else
                        ln = -v - 1;
                }
                L.slotn[t] = sl;
                L.link[t] = ln;
                chain |= sl < 0;
            }
        }
        // an entrant evicted within its block passes its slot on to the
        // entrant that evicted it: resolve the chains by pointer jumping (a
        // link points to an earlier entrant, so a chain of at most kCapB
        // entrants resolves within log2(kCapB) + 1 rounds; the bound only
        // guards the loop)
        if (__syncthreads_or(chain)) {
            for (int round = 0; round < 16; ++round) {
                bool un = false;
                int sl[U], ln[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int t = u * kSelT + tid;
                    sl[u] = -1;
                    ln[u] = -1;
                    if (t < e && L.slotn[t] < 0) {
                        un = true;
                        const int l = L.link[t];
                        sl[u] = L.slotn[l];
                        ln[u] = L.link[l];
                    }
                }
                if (!__syncthreads_or(un)) break;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int t = u * kSelT + tid;
                    if (t < e && L.slotn[t] < 0) {
                        if (sl[u] >= 0)
                            L.slotn[t] = sl[u];
                        else
                            L.link[t] = ln[u];
                    }
                }
                __syncthreads();
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = u * kSelT + tid;
            if (t < e && L.nU[t] < cap) Ts[L.nU[t]] = L.slotn[t];
        }
        __syncthreads();
        s = snew;
        buf ^= 1;
    }
    bufo = buf;
    return s;
}

// Cap one candidate stream (cap above LEKF_CAP_LDS) with the whole workgroup
// and write the kept entries in slot order: emit(slot, candidate).  Uniform
// call; ends with a barrier.
template <class KeyAt, class Emit>
__device__ int cap_stream(SelLds& S, const CapGlobal& G, KeyAt keyat, Emit emit, int n, int cap,
                          int tid)
{
    int buf = 0;
    const int kept = cap_slots(S.cap, G, keyat, n, cap, tid, buf);
    for (int r = tid; r < kept; r += kSelT) {
        const int sl = G.slot[(size_t)buf * cap + r];
        if ((unsigned)sl < (unsigned)kept) emit(sl, G.pos[(size_t)buf * cap + r]);
    }
    __syncthreads();
    return kept;
}

// ---------------------------------------------------------------------------
// The cap by one wave (caps up to LEKF_CAP_LDS), fed with the candidates of one
// bucket stream in scan order.
//
// The kept set S (the cap smallest (key, scan position) of the stream so far) is
// held ascending in key[], with each entry's storage slot in slot[]; so[s]
// (caller's memory) is the candidate in storage slot s.  The first cap candidates
// fill slots 0..cap-1: only their positions are kept until the cap-th arrives, then
// they are sorted in by batches.  A later candidate can enter only if its key is
// below the key tau of S's last entry (an earlier candidate with an equal key
// precedes it), and tau only falls, so the caller filters candidates by any bound
// that keeps every key below tau, into a queue, and up to kWcB = 224 queued
// candidates are evaluated exactly (four per lane, their long chains overlapping)
// and merged at once:
// * a candidate enters iff fewer than cap of S and of the earlier queued
//   candidates precede it.  All of S precedes it in scan order, so its count there
//   is c1, the number of keys <= its key; the block's candidates are ranked by key
//   (a counting sort over the leading bits of the keys' range), and where c1 and the
//   rank together reach cap the earlier ones among those ranked before are counted
//   as a set of scan positions;
// * the entrants are counted per c1: a scan of the counts over S from the top gives
//   every entry's move;
// * of S and the entrants the top e leave; the i-th entrant in scan order takes the
//   slot of the i-th largest entry that left: the reference evicts the current last
//   entry each time, and the last key only falls; an entrant that leaves in its own
//   block hands its slot on (pointer jumping).
// Bound by VALU issue: 67% busy at three waves per SIMD, 52 k vector and 18 k scalar
// instructions a stream (radar 256 x 256 x 60, two streams of 12.6 k candidates per point).
// Against blocks of 64 sorted across the lanes with every candidate evaluated exactly as
// it was scanned, the radar 128 x 128 x 60 selection takes 251 instead of 401 ms per cycle,
// the GFS-sized grid's list_cap_wave 22 instead of 33 ms.
// ---------------------------------------------------------------------------

// order of the lanes' LDS traffic within the wave (no cross-wave sharing)
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Candidates per block, at most kWcU per lane.  The LDS decides how many waves hide
// each other's latencies: 13,440 bytes a wave are 21 granules (1280 bytes) for two,
// six such workgroups per CU, three waves per SIMD.
constexpr int kWcU = 4;
constexpr int kWcB = 224;

struct __align__(16) WaveCap {
    unsigned long long key[LEKF_CAP_LDS];  // while S fills: the positions, in the upper half
    unsigned cnt[LEKF_CAP_LDS / 2];        // 16-bit counts, and what comes after them in a block
    unsigned short slot[LEKF_CAP_LDS];
    int qp[kWcB + 64];                     // queued candidates, scan order
};
static_assert(sizeof(WaveCap) == 13440, "LDS per wave of the cap");
constexpr unsigned short kWcOwn = 0x8000, kWcNone = 0xffff;

// Positions of the first cap candidates.  When the fill has sorted the first lim of
// them their keys end at byte 8 lim and the positions still to come begin at byte
// 4 LEKF_CAP_LDS + 4 lim, so none is overwritten before it is read.
__device__ __forceinline__ int* wc_fill_pos(WaveCap& L)
{
    return (int*)(L.key + LEKF_CAP_LDS / 2);
}

struct WcState {
    int n;                   // stream candidates so far (exact up to cap)
    int m;                   // sorted prefix of S while it fills
    int q;                   // queued candidates
    unsigned long long tau;  // key of S's last entry (once m = cap)
};

__device__ __forceinline__ int wave_scan(int v)  // inclusive sum over the lanes up to this one
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

__device__ __forceinline__ unsigned wave_scan_or(unsigned v)  // the same, by or
{
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned dpp_max(unsigned v)
{
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    return o > v ? o : v;
}
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
    v = dpp_max<0x111, 0xf>(v);
    v = dpp_max<0x112, 0xf>(v);
    v = dpp_max<0x114, 0xf>(v);
    v = dpp_max<0x118, 0xf>(v);
    v = dpp_max<0x142, 0xa>(v);
    v = dpp_max<0x143, 0xc>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ unsigned wave_min(unsigned v) { return ~wave_max(~v); }

// The counts: LEKF_CAP_LDS of 16 bits (no count passes kWcB), added to in pairs.
__device__ __forceinline__ void wc_zero(WaveCap& L, int lane)
{
#pragma unroll
    for (int j = 0; j < LEKF_CAP_LDS / 512; ++j)
        reinterpret_cast<uint4*>(L.cnt)[j * 64 + lane] = make_uint4(0, 0, 0, 0);
}
__device__ __forceinline__ int wc_count(WaveCap& L, int i)  // returns the count before
{
    const int sh = (i & 1) * 16;
    return (int)((atomicAdd(&L.cnt[i >> 1], 1u << sh) >> sh) & 0xffffu);
}

// One block: np <= kWcB candidates (positions src[0 .. np), scan order) join S.
// fill < 0: S is full, queued candidates against tau; else S's first fill entries are
// sorted and the candidates are its entries fill .. fill + np - 1, in slots of that
// number.  eval(p, ok): the key of the candidate at position p, ok: it is a stream
// candidate (the fill's are).  Returns S's new last key.
template <class Eval>
__device__ __forceinline__ unsigned long long wc_block(WaveCap& L, int* so, const int* src, int np,
                                                       int fill, int cap, int lane,
                                                       unsigned long long tau, Eval eval)
{
    const bool full = fill < 0;
    const int n = full ? cap : fill;         // entries of S
    const int lim = full ? cap : fill + np;  // and after the block
    int p[kWcU], c1[kWcU], t[kWcU], rank[kWcU];
    unsigned long long y[kWcU];
    bool ent[kWcU];
#pragma unroll
    for (int u = 0; u < kWcU; ++u) p[u] = u * 64 + lane < np ? src[u * 64 + lane] : -1;
    wave_sync();
    wc_zero(L, lane);
    int nlive = 0;
    unsigned hmin = ~0u, hmax = 0u;
#pragma unroll
    for (int u = 0; u < kWcU; ++u) {
        bool ok = false;
        y[u] = ~0ull;
        if (p[u] >= 0) y[u] = eval(p[u], ok);
        ent[u] = p[u] >= 0 && (full ? ok && y[u] < tau : true);
        nlive += __popcll(__ballot(ent[u]));
        const unsigned h = (unsigned)(y[u] >> 32);
        if (ent[u]) {
            hmin = h < hmin ? h : hmin;
            hmax = h > hmax ? h : hmax;
        }
    }
    if (nlive == 0) return tau;
    // rank by key: counting sort over the leading bits of the keys' range, then a look
    // at the candidates of the same count
    {
        const unsigned long long k0 = (unsigned long long)wave_min(hmin) << 32;
        const unsigned span = wave_max(hmax) - (unsigned)(k0 >> 32);
        const int sh = span ? 54 - __builtin_clz(span) : 22;  // (span + 1) 2^32 - 1 >> sh < 1024
        int g[kWcU], tick[kWcU], base[kWcU], mem[kWcU], big = 1;
        wave_sync();
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            g[u] = ent[u] ? (int)((y[u] - k0) >> sh) : 0;
            tick[u] = ent[u] ? wc_count(L, g[u]) : 0;
        }
        wave_sync();
        unsigned short* cnt = (unsigned short*)L.cnt;  // counts to the ranks they start at
        int run = 0;
        for (int lo = 0; lo < LEKF_CAP_LDS; lo += 256) {
            int cn[4], pin[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) cn[j] = cnt[lo + 64 * j + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) pin[j] = wave_scan(cn[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                cnt[lo + 64 * j + lane] = (unsigned short)(run + pin[j] - cn[j]);
                run += __builtin_amdgcn_readlane(pin[j], 63);
            }
        }
        wave_sync();
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            base[u] = cnt[g[u]];
            mem[u] = ent[u] ? (g[u] + 1 < LEKF_CAP_LDS ? (int)cnt[g[u] + 1] : nlive) - base[u] : 0;
            big = mem[u] > big ? mem[u] : big;
            rank[u] = base[u];
        }
        wave_sync();
        unsigned long long* ekey = (unsigned long long*)L.cnt;  // the counts are spent
        unsigned char* eidx = (unsigned char*)(ekey + kWcB);
#pragma unroll
        for (int u = 0; u < kWcU; ++u)
            if (mem[u] > 1) {
                ekey[base[u] + tick[u]] = y[u];
                eidx[base[u] + tick[u]] = (unsigned char)(u * 64 + lane);
            }
        wave_sync();
        for (int j = 0; __ballot(big > 1 && j < big); ++j)
#pragma unroll
            for (int u = 0; u < kWcU; ++u)
                if (j < mem[u] && mem[u] > 1) {
                    const unsigned long long x = ekey[base[u] + j];
                    rank[u] += x < y[u] || (x == y[u] && (int)eidx[base[u] + j] < u * 64 + lane);
                }
        wave_sync();
    }
    // entries of S before each candidate
    {
        int lo[kWcU], hi[kWcU];
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            lo[u] = 0;
            hi[u] = ent[u] ? n : 0;
        }
        for (int w = n; w > 0; w >>= 1)
#pragma unroll
            for (int u = 0; u < kWcU; ++u) {
                const int mid = (lo[u] + hi[u]) >> 1;
                const bool le = L.key[mid < n ? mid : 0] <= y[u];
                if (lo[u] < hi[u]) {
                    lo[u] = le ? mid + 1 : lo[u];
                    hi[u] = le ? hi[u] : mid;
                }
            }
#pragma unroll
        for (int u = 0; u < kWcU; ++u) c1[u] = lo[u];
    }
    int e = nlive;
    if (full) {
        // a live candidate enters if fewer than cap of S and of the live candidates
        // before it precede it; rank bounds the latter
        bool amb = false;
        int lt[kWcU], before = 0;
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            const unsigned long long m = __ballot(ent[u]);
            const int r = before + __popcll(m & lane_lt(lane));
            lt[u] = r < rank[u] ? r : rank[u];
            amb |= ent[u] && c1[u] + lt[u] >= cap;
            before += __popcll(m);
        }
        if (__ballot(amb)) {
            // in rank order, four candidates per lane: the set of scan positions
            // ranked before each (their bits are distinct), and of it those earlier
            unsigned char* sidx = (unsigned char*)L.cnt;
            unsigned short* c2 = (unsigned short*)(L.cnt + 64);
#pragma unroll
            for (int u = 0; u < kWcU; ++u)
                if (ent[u]) sidx[rank[u]] = (unsigned char)(u * 64 + lane);
            wave_sync();
            const unsigned ids = L.cnt[lane];
            unsigned own[8], ex[8];
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                own[d] = 0;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = (ids >> (8 * v)) & 255;
                    if (4 * lane + v < nlive && (i >> 5) == d) own[d] |= 1u << (i & 31);
                }
                ex[d] = wave_scan_or(own[d]) & ~own[d];
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = (ids >> (8 * v)) & 255;
                int c = 0;
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    const unsigned lower = (i >> 5) > d ? ~0u : (i >> 5) == d ? (1u << (i & 31)) - 1 : 0u;
                    c += __popc(ex[d] & lower);
                    if ((i >> 5) == d) ex[d] |= 1u << (i & 31);
                }
                if (4 * lane + v < nlive) c2[4 * lane + v] = (unsigned short)c;
            }
            wave_sync();
            // the entrants, and their ranks among themselves
            bool in[kWcU];
            e = 0;
#pragma unroll
            for (int u = 0; u < kWcU; ++u) {
                in[u] = ent[u] && c1[u] + (int)c2[ent[u] ? rank[u] : 0] < cap;
                e += __popcll(__ballot(in[u]));
            }
            if (e == 0) return tau;
            wave_sync();
            if (e < nlive) {
                L.cnt[lane] = 0;
                wave_sync();
#pragma unroll
                for (int u = 0; u < kWcU; ++u)
                    if (in[u]) sidx[rank[u]] = 1;
                wave_sync();
                const unsigned fl = L.cnt[lane];
                const int own4 = __popc(fl);
                int r = wave_scan(own4) - own4;
                unsigned short* re = c2;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    re[4 * lane + v] = (unsigned short)r;
                    r += (fl >> (8 * v)) & 1;
                }
                wave_sync();
#pragma unroll
                for (int u = 0; u < kWcU; ++u) {
                    ent[u] = in[u];
                    if (in[u]) rank[u] = re[rank[u]];
                }
                wave_sync();
            }
        }
    }
    {
        int before = 0;
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            const unsigned long long m = __ballot(ent[u]);
            t[u] = before + __popcll(m & lane_lt(lane));  // rank among the entrants, scan order
            before += __popcll(m);
        }
    }
    // entrants per c1; then, from the top down, 256 entries of S at a time: entry i
    // moves up by the entrants with c1 <= i (writes only reach entries that have been
    // read)
    wc_zero(L, lane);
    wave_sync();
#pragma unroll
    for (int u = 0; u < kWcU; ++u)
        if (ent[u]) (void)wc_count(L, c1[u]);
    wave_sync();
    const unsigned short* at = (const unsigned short*)L.cnt;
    unsigned short* ev = (unsigned short*)L.qp;  // entries that left, ascending: slot, or
                                                 // kWcOwn + entrant (these candidates are read)
    for (int lo = (full ? n - 1 : n) & ~255, left = e; lo >= 0 && left > 0; lo -= 256) {
        int cn[4], shift[4];
        unsigned long long k[4];
        unsigned short s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = lo + 64 * j + lane;
            cn[j] = at[i];
            k[j] = L.key[i];
            s[j] = L.slot[i];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) shift[j] = wave_scan(cn[j]);
        int tot = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int w = __builtin_amdgcn_readlane(shift[j], 63);
            shift[j] += tot;
            tot += w;
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = lo + 64 * j + lane;
            const int ni = i + left - tot + shift[j];
            if (i < n && ni > i) {
                if (ni < lim) {
                    L.key[ni] = k[j];
                    L.slot[ni] = s[j];
                } else {
                    ev[ni - lim] = s[j];
                }
            }
        }
        left -= tot;
        wave_sync();
    }
    if (!full) {
#pragma unroll
        for (int u = 0; u < kWcU; ++u)
            if (ent[u]) {
                const int q = c1[u] + rank[u];
                L.key[q] = y[u];
                L.slot[q] = (unsigned short)(fill + t[u]);
                so[fill + t[u]] = p[u];
            }
        wave_sync();
        return L.key[lim - 1];
    }
#pragma unroll
    for (int u = 0; u < kWcU; ++u)
        if (ent[u]) {
            const int q = c1[u] + rank[u];
            if (q < cap)
                L.key[q] = y[u];
            else
                ev[q - cap] = (unsigned short)(kWcOwn | t[u]);
        }
    wave_sync();
    unsigned short* slotn = (unsigned short*)L.cnt;  // the counts are spent
    unsigned short* link = slotn + kWcB;
    int sl[kWcU], ln[kWcU];
    bool open = false;
#pragma unroll
    for (int u = 0; u < kWcU; ++u) {
        sl[u] = 0;
        ln[u] = 0;
        if (ent[u]) {
            const int v = ev[e - 1 - t[u]];
            const bool own = (v & kWcOwn) != 0;
            sl[u] = own ? -1 : v;
            ln[u] = v & ~kWcOwn;
            open |= own;
            slotn[t[u]] = own ? kWcNone : (unsigned short)v;
            link[t[u]] = (unsigned short)ln[u];
        }
    }
    wave_sync();
    // chains of at most kWcB entrants: 8 doublings
    for (int round = 0; round < 8 && __ballot(open); ++round) {
        int s2[kWcU], l2[kWcU];
#pragma unroll
        for (int u = 0; u < kWcU; ++u) {
            s2[u] = slotn[sl[u] < 0 ? ln[u] : 0];
            l2[u] = link[sl[u] < 0 ? ln[u] : 0];
        }
        wave_sync();
        open = false;
#pragma unroll
        for (int u = 0; u < kWcU; ++u)
            if (sl[u] < 0) {
                if (s2[u] != kWcNone)
                    sl[u] = s2[u];
                else
                    ln[u] = l2[u];
                open |= sl[u] < 0;
                slotn[t[u]] = sl[u] < 0 ? kWcNone : (unsigned short)sl[u];
                link[t[u]] = (unsigned short)ln[u];
            }
        wave_sync();
    }
#pragma unroll
    for (int u = 0; u < kWcU; ++u)
        if (ent[u] && c1[u] + rank[u] < cap && sl[u] >= 0) {
            L.slot[c1[u] + rank[u]] = (unsigned short)sl[u];
            so[sl[u]] = p[u];
        }
    wave_sync();
    return L.key[cap - 1];
}

// The same block of at most 64 candidates, one per lane, for small caps and short streams,
// where the counts over LEKF_CAP_LDS places and the scans over them would cost more than
// the candidates: they are sorted across the lanes by (key, lane), and the entries of S move
// up 64 at a time, one entrant after the other counted.
__device__ __forceinline__ void wc_sort64(unsigned long long& k, int& id, int lane)
{
#pragma unroll
    for (int sz = 2; sz <= 64; sz <<= 1) {
#pragma unroll
        for (int j = sz >> 1; j > 0; j >>= 1) {
            const unsigned lo = (unsigned)lane_xor((int)(unsigned)k, j, lane);
            const unsigned hi = (unsigned)lane_xor((int)(unsigned)(k >> 32), j, lane);
            const unsigned long long ok = ((unsigned long long)hi << 32) | lo;
            const int oid = lane_xor(id, j, lane);
            const bool up = (lane & sz) == 0;
            const bool lower = (lane & j) == 0;
            const bool oless = ok < k || (ok == k && oid < id);
            if (lower == up ? oless : !oless) {
                k = ok;
                id = oid;
            }
        }
    }
}

// Entries 0 .. n-1 of S move up by the entrants placed before them (lanes with ent, at
// count c1 of the old entries, ascending: before entry i iff c1 <= i); an entry that lands
// at lim or above goes to ev (its slot).  Windows of 64 go top down, so a window's writes
// only reach entries that have moved.
__device__ __forceinline__ void wc_shift64(WaveCap& L, int* ev, int n, int lim, bool ent, int c1,
                                           int lane)
{
    const unsigned long long em = __ballot(ent);
    if (!em || n <= 0) return;
    const int c1min = __builtin_amdgcn_readlane(c1, __builtin_ctzll(em));
    for (int lo = ((n - 1) >> 6) << 6; lo >= 0 && lo + 64 > c1min; lo -= 64) {
        const int i = lo + lane;
        unsigned long long k = 0;
        int s = 0;
        if (i < n) {
            k = L.key[i];
            s = L.slot[i];
        }
        int up = __popcll(__ballot(ent && c1 < lo));
        for (unsigned long long w = __ballot(ent && c1 >= lo && c1 < lo + 64); w; w &= w - 1)
            up += lane >= __builtin_amdgcn_readlane(c1, __builtin_ctzll(w)) - lo ? 1 : 0;
        if (i < n && up > 0) {
            if (i + up < lim) {
                L.key[i + up] = k;
                L.slot[i + up] = (unsigned short)s;
            } else {
                ev[i + up - lim] = s;
            }
        }
    }
}

template <class Eval>
__device__ __forceinline__ unsigned long long wc_block64(WaveCap& L, int* so, const int* src,
                                                         int np, int fill, int cap, int lane,
                                                         unsigned long long tau, Eval eval)
{
    const bool full = fill < 0;
    const int n = full ? cap : fill;         // entries of S
    const int lim = full ? cap : fill + np;  // and after the block
    int* ev = (int*)L.cnt;  // entries that left, ascending: slot, or -(entrant + 1)
    int* slotn = ev + 64;
    int* link = ev + 128;
    const int p = lane < np ? src[lane] : -1;
    wave_sync();
    bool ok = false;
    unsigned long long y = ~0ull;
    if (p >= 0) y = eval(p, ok);
    const bool live = p >= 0 && (full ? ok && y < tau : true);
    const int nlive = __popcll(__ballot(live));
    if (nlive == 0) return tau;
    // sorted by (key, lane), the live candidates first
    unsigned long long sk = live ? y : ~0ull;
    int sid = live ? lane : lane + 64;
    wc_sort64(sk, sid, lane);
    sid &= 63;
    const bool slive = lane < nlive;
    const int ps = __shfl(p, sid, 64);
    int c1 = 0;  // entries of S before it
    {
        int lo = 0, hi = slive ? n : 0;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (L.key[mid] <= sk)
                lo = mid + 1;
            else
                hi = mid;
        }
        c1 = lo;
    }
    wave_sync();
    if (!full) {
        wc_shift64(L, ev, n, lim, slive, c1, lane);
        wave_sync();
        if (slive) {
            L.key[c1 + lane] = sk;
            L.slot[c1 + lane] = (unsigned short)(fill + sid);
            so[fill + sid] = ps;
        }
        wave_sync();
        return L.key[lim - 1];
    }
    // earlier (in scan order) live candidates sorted before this one
    const unsigned long long own = slive ? 1ull << sid : 0ull;
    unsigned long long pm = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_up(pm, d, 64);
        if (lane >= d) pm |= o;
    }
    const int c2 = __popcll(pm & ~own & lane_lt(sid));
    const bool ent = slive && c1 + c2 < cap;
    const unsigned long long em = __ballot(ent);
    const int e = __popcll(em);
    if (e == 0) return tau;
    const int at = c1 + __popcll(em & lane_lt(lane));  // position in S and the entrants
    // scan-order index of each entrant: its flag back to the candidate's lane
    const unsigned long long eo =
        __ballot(__builtin_amdgcn_ds_permute(sid << 2, ent ? 1 : 0) != 0);
    const int t = __popcll(eo & lane_lt(sid));
    wc_shift64(L, ev, cap, cap, ent, c1, lane);
    wave_sync();
    if (ent) {
        if (at < cap)
            L.key[at] = sk;
        else
            ev[at - cap] = -(t + 1);
    }
    wave_sync();
    int sl = -1, ln = -1;
    if (ent) {
        const int v = ev[e - 1 - t];
        if (v >= 0)
            sl = v;
        else
            ln = -v - 1;
        slotn[t] = sl;
        link[t] = ln;
    }
    wave_sync();
    // chains of at most 64 entrants: 6 doublings
    for (int round = 0; round < 6 && __ballot(ent && sl < 0); ++round) {
        int s2 = -1, l2 = -1;
        if (ent && sl < 0) {
            s2 = slotn[ln];
            l2 = link[ln];
        }
        wave_sync();
        if (ent && sl < 0) {
            if (s2 >= 0)
                sl = s2;
            else
                ln = l2;
            slotn[t] = sl;
            link[t] = ln;
        }
        wave_sync();
    }
    if (ent && at < cap && sl >= 0) {
        L.slot[at] = (unsigned short)sl;
        so[sl] = ps;
    }
    wave_sync();
    return L.key[cap - 1];
}

// A chunk of the stream: lane l's candidate p enters the fill or the queue iff in
// (while S fills every stream candidate; then at least those with a key below tau).
__device__ __forceinline__ void wc_push(WaveCap& L, WcState& S, bool in, int p, int cap, int lane)
{
    const unsigned long long m = __ballot(in);
    if (!m) return;
    const int cnt = __popcll(m), rank = __popcll(m & lane_lt(lane));
    const int room = S.n < cap ? cap - S.n : 0;  // the fill's share
    if (in) {
        if (rank < room)
            wc_fill_pos(L)[S.n + rank] = p;
        else
            L.qp[S.q + rank - room] = p;
    }
    const int f = cnt < room ? cnt : room;
    S.n += f;
    S.q += cnt - f;
    wave_sync();
}

// Blocks that are due: the fill's once S has cap entries, the queue's when a block's
// candidates wait (kWcB, SMALL: 64), or any with last.
template <bool SMALL, class Eval>
__device__ __forceinline__ void wc_service(WaveCap& L, int* so, WcState& S, int cap, int lane,
                                           bool last, Eval eval)
{
    constexpr int B = SMALL ? 64 : kWcB;
    while (S.n >= cap) {
        const bool filling = S.m < cap;
        if (!filling && S.q < B && !(last && S.q > 0)) break;
        const int have = filling ? cap - S.m : S.q;
        const int np = have < B ? have : B;
        const int* src = filling ? wc_fill_pos(L) + S.m : L.qp;
        const int fill = filling ? S.m : -1;
        if constexpr (SMALL)
            S.tau = wc_block64(L, so, src, np, fill, cap, lane, S.tau, eval);
        else
            S.tau = wc_block(L, so, src, np, fill, cap, lane, S.tau, eval);
        if (filling) {
            S.m += np;
        } else {
            // the rest of the queue (fewer than 64) moves to its front
            S.q -= np;
            int o = 0;
            if (lane < S.q) o = L.qp[B + lane];
            wave_sync();
            if (lane < S.q) L.qp[lane] = o;
            wave_sync();
        }
    }
}

// Persistent selection: workgroup g handles points g, g + gridDim.x, ...
// Each candidate of a point is evaluated once.  Without a cap the accepted
// candidates are written in scan order.  With a cap each bucket's accepted
// candidates go, in scan order, to the bucket's stream in the workgroup's
// scratch (rdiag bits, obs, rho); a stream within the cap is written as it
// is, a longer one through cap_stream in slot order, bucket after bucket.
__global__ __launch_bounds__(kSelT) void reg_select(RegionalArgs A, long npt)
{
    __shared__ SelLds S;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    const int nij = A.nx * A.ny;
    const int nb = A.nbkt;
    const int cap = A.nobs_max;
    const size_t sbase = (size_t)blockIdx.x * (size_t)nb * (size_t)A.slot_cap;
    unsigned long long* skey = A.s_key + sbase;
    int* sob = A.s_ob + sbase;
    double* srho = A.s_rho + sbase;
    CapGlobal G;
    G.key = A.g_key ? A.g_key + (size_t)blockIdx.x * 2 * cap : nullptr;
    G.pos = A.g_pos ? A.g_pos + (size_t)blockIdx.x * 2 * cap : nullptr;
    G.slot = A.g_slot ? A.g_slot + (size_t)blockIdx.x * 2 * cap : nullptr;

    for (long pi = blockIdx.x; pi < npt; pi += gridDim.x) {
        const long b = A.pt_begin + pi;  // global point = lev * nij + ij
        const int lev = (int)(b / nij), ij = (int)(b % nij);
        const double ri = (double)(ij % A.nx + 1), rj = (double)(ij / A.nx + 1), rz = A.zlev[lev];
        int imin = (int)floor(ri - A.dlon_zero), imax = (int)ceil(ri + A.dlon_zero);
        int jmin = (int)floor(rj - A.dlat_zero), jmax = (int)ceil(rj + A.dlat_zero);
        if (imin < 1) imin = 1;
        if (imax > A.nx) imax = A.nx;
        if (jmin < 1) jmin = 1;
        if (jmax > A.ny) jmax = A.ny;
        const int nseg = (imin > imax || jmin > jmax) ? 0 : jmax - jmin + 1;
        if (tid == 0) {
            int acc = 0;
            for (int s = 0; s < nseg; ++s) {
                const int j = jmin + s;  // 1-based row
                // cellcum = inclusive cumulative count through cell (i, j), row-major
                const long rowbase = (long)(j - 1) * A.nx;
                const int beg = (imin > 1) ? A.cellcum[rowbase + imin - 2]
                                           : (rowbase > 0 ? A.cellcum[rowbase - 1] : 0);
                const int end = A.cellcum[rowbase + imax - 1];
                S.seg_beg[s] = beg;
                S.seg_pre[s] = acc;
                acc += end - beg;
            }
            S.seg_pre[nseg] = acc;
        }
        __syncthreads();
        const int ncand = S.seg_pre[nseg];
        const long obase = A.list_off[b] - A.list_base;  // relative to this chunk's list buffer

        // evaluate every candidate once; scan position q = q0 + tid
        int nacc = 0;
        int bcnt[LEKF_REG_NB];
#pragma unroll
        for (int t = 0; t < LEKF_REG_NB; ++t) bcnt[t] = 0;
        int seg = 0;
        for (int q0 = 0; q0 < ncand; q0 += kSelT) {
            const int q = q0 + tid;
            const int o = q < ncand ? cand_obs(S, nseg, q, seg) : -1;
            Cand c;
            c.ok = false;
            c.b = 0;
            if (o >= 0) c = eval_rec(A, load_obs(A, o), o, ri, rj, rz);
            unsigned long long m[LEKF_REG_NB];
#pragma unroll
            for (int t = 0; t < LEKF_REG_NB; ++t)
                m[t] = __ballot(c.ok && (cap <= 0 || c.b == t));
            if (lane == 0)
#pragma unroll
                for (int t = 0; t < LEKF_REG_NB; ++t) S.wcnt[wv][t] = __popcll(m[t]);
            __syncthreads();
            int pos = -1;
            if (cap <= 0) {
                int before = 0, tot = 0;
                for (int w = 0; w < kSelW; ++w) {
                    const int cw = S.wcnt[w][0];
                    before += w < wv ? cw : 0;
                    tot += cw;
                }
                pos = nacc + before + __popcll(m[0] & lane_lt(lane));
                nacc += tot;
            } else {
#pragma unroll
                for (int t = 0; t < LEKF_REG_NB; ++t) {
                    int before = 0, tot = 0;
                    for (int w = 0; w < kSelW; ++w) {
                        const int cw = S.wcnt[w][t];
                        before += w < wv ? cw : 0;
                        tot += cw;
                    }
                    if (c.ok && c.b == t) pos = bcnt[t] + before + __popcll(m[t] & lane_lt(lane));
                    bcnt[t] += tot;
                }
            }
            __syncthreads();
            if (c.ok) {
                if (cap <= 0) {
                    A.loc_idx[obase + pos] = c.o;
                    A.loc_rho[obase + pos] = c.rho;
                } else {
                    const size_t w = (size_t)c.b * (size_t)A.slot_cap + (size_t)pos;
                    skey[w] = c.bits;
                    sob[w] = c.o;
                    srho[w] = c.rho;
                }
            }
        }
        __syncthreads();
        if (cap > 0) {
            nacc = 0;
            for (int t = 0; t < nb; ++t) {
                const int n = bcnt[t];
                const size_t so = (size_t)t * (size_t)A.slot_cap;
                int* oi = A.loc_idx + obase + nacc;
                double* orh = A.loc_rho + obase + nacc;
                if (n <= cap) {
                    for (int i = tid; i < n; i += kSelT) {
                        oi[i] = sob[so + i];
                        orh[i] = srho[so + i];
                    }
                    nacc += n;
                } else {
                    nacc += cap_stream(
                        S, G, [&](int i) { return skey[so + i]; },
                        [&](int slot, int i) {
                            oi[slot] = sob[so + i];
                            orh[slot] = srho[so + i];
                        },
                        n, cap, tid);
                }
            }
        }
        if (tid == 0) {
            A.loc_off[b] = obase;
            A.loc_cnt[b] = nacc;
        }
        __syncthreads();
    }
}

// Capped selection with the kept sets in LDS (0 < nobs_max <= LEKF_CAP_LDS):
// persistent, one point per workgroup, wave t caps bucket t's stream (NW =
// nbkt waves).  A bucket's candidates in the point's rectangle are, row by
// row, one contiguous range of the bucket-by-bucket obs copy, in the
// reference's scan order restricted to the bucket.  The scan reads a 16-byte
// FP32 record per candidate and decides in FP32 where its error bound allows:
// candidates within the bound of the cutoff while S fills are evaluated exactly,
// later ones whose key may be below tau go to the wave's queue and are evaluated
// exactly there (eval_rec), so the lists are the reference's.  They are written
// bucket by bucket in slot order, rho recomputed from the kept obs.
constexpr int kTileX = 16, kTileY = 8;  // columns of a selection tile

//
// Forms.  kDense: each row's candidates in chunks of their own.  kFewRows: rows of a few
// candidates, several in a chunk.  kSmallCap: the same, and blocks of 64.
constexpr int kDense = 0, kFewRows = 1, kSmallCap = 2;

template <int NW, int FORM>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3)))
void reg_select_wave(RegionalArgs A, long npt)
{
    __shared__ WaveCap L[NW];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int nij = A.nx * A.ny;
    const int cap = A.nobs_max;
    const int* cc = A.bcc + (size_t)wv * nij;
    int bs = 0;  // bucket wv's first position in the bucket-by-bucket copy
    for (int u = 0; u < wv; ++u) bs += A.bcc[(size_t)u * nij + nij - 1];
    WaveCap& W = L[wv];
    int* so = A.wc_so + ((size_t)blockIdx.x * NW + wv) * LEKF_CAP_LDS;  // slot -> position
    const double r2cut = kNdMax * A.sigma_h * A.sigma_h * (1.0 + 1e-9);
    // the bucket's smallest err^2 (NaN for an empty bucket: never used)
    const double e2min = A.err2_min ? __longlong_as_double((long long)A.err2_min[wv]) : 0.0;
    const double ish2 = 1.0 / (A.sigma_h * A.sigma_h);
    const float cx = (float)(A.dx * A.dx * ish2), cy = (float)(A.dy * A.dy * ish2);
    const float cv = (float)(1.0 / (A.sigma_v * A.sigma_v));
    // rounding of a horizontal coordinate difference in FP32, in units of sigma_h
    const double eh = (A.nx > A.ny ? A.nx : A.ny) * 1.2e-7 *
                      (A.dx > A.dy ? A.dx : A.dy) / A.sigma_h;
    // the position's record, evaluated exactly
    auto load_rec = [&](int p) {
        const double2 rij = *reinterpret_cast<const double2*>(A.brec + 4 * (size_t)p);
        const double2 zer = *reinterpret_cast<const double2*>(A.brec + 4 * (size_t)p + 2);
        return ObsRec{rij.x, rij.y, zer.x, zer.y, wv};
    };

    // XCD-aware tile order: workgroup w runs on XCD w % 8 (round-robin
    // dispatch); the XCD's workgroups take the points of one kTileX x kTileY
    // block of columns at one level together, so the obs of the block's
    // rectangles stay in that XCD's L2.  Group x (x < ng = min(8, grid)) takes
    // the tiles t = x (mod ng), its workgroups the tile's points in turn.
    const int ng = gridDim.x < 8 ? (int)gridDim.x : 8;
    const int xcd = (int)blockIdx.x % ng, wj = (int)blockIdx.x / ng;
    const int nwg = ((int)gridDim.x - xcd + ng - 1) / ng;
    const int tnx = (A.nx + kTileX - 1) / kTileX, tny = (A.ny + kTileY - 1) / kTileY;
    const long tpl = (long)tnx * tny;  // tiles per level
    const long bend = A.pt_begin + npt;
    const long t_first = (A.pt_begin / nij) * tpl, t_last = ((bend - 1) / nij + 1) * tpl - 1;
    const long t0 = t_first + ((xcd - t_first % ng) + ng) % ng;
    for (long q = wj;; q += nwg) {
        const long t = t0 + (q / (kTileX * kTileY)) * ng;
        if (t > t_last) break;
        const int w = (int)(q % (kTileX * kTileY));
        const int lev = (int)(t / tpl), tl = (int)(t % tpl);
        const int ix = (tl % tnx) * kTileX + w % kTileX, iy = (tl / tnx) * kTileY + w / kTileX;
        if (ix >= A.nx || iy >= A.ny) continue;
        const int ij = iy * A.nx + ix;
        const long b = (long)lev * nij + ij;  // global point
        if (b < A.pt_begin || b >= bend) continue;
        const double ri = (double)(ix + 1), rj = (double)(iy + 1), rz = A.zlev[lev];
        int imin = (int)floor(ri - A.dlon_zero), imax = (int)ceil(ri + A.dlon_zero);
        int jmin = (int)floor(rj - A.dlat_zero), jmax = (int)ceil(rj + A.dlat_zero);
        if (imin < 1) imin = 1;
        if (imax > A.nx) imax = A.nx;
        if (jmin < 1) jmin = 1;
        if (jmax > A.ny) jmax = A.ny;
        const float fri = (float)(ix + 1), frj = (float)(iy + 1), frz = (float)rz;
        // bound of the FP32 nd's error for nd up to the cutoff (sqrt 13.4 < 3.7):
        // 2 sqrt(nd) (e_x + e_y + e_z) + the squares + the arithmetic's 1e-5
        const double ev = (fabs(rz) + 4.0 * A.sigma_v) * 1.2e-7 / A.sigma_v;
        const double es = 2.0 * eh + ev;
        const float em = (float)(7.4 * es + es * es + 1.0e-4);
        const float nd_out = (float)kNdMax + em, nd_in = (float)kNdMax - em;
        float l2tau = 3.0e38f;  // log2 tau and the bound
        WcState S{0, 0, 0, ~0ull};
        auto eval = [&](int p, bool& ok) {
            const Cand c = eval_rec(A, load_rec(p), p, ri, rj, rz);
            ok = c.ok;
            return c.bits;
        };
        bool fin = imin > imax;
        for (int j0 = jmin;; j0 += 64) {
            fin |= j0 > jmax;
            const int nr = fin ? 0 : (jmax - j0 + 1 < 64 ? jmax - j0 + 1 : 64);
            int beg = 0, len = 0;
            if (lane < nr) {
                // the row's cells that can hold an obs within the cutoff: a
                // cell's obs lie on its side of the faces at i +- 0.5, so one
                // whose nearest face is beyond the cutoff radius holds none
                // (nd >= nd_h^2 > kNdMax); a 1e-9 margin covers rounding
                const int j = j0 + lane;
                const double dyg = fmax(0.0, fabs((double)j - rj) - 0.5) * A.dy;
                const double rem = r2cut - dyg * dyg;
                int ilo = imin, ihi = imax;
                if (rem < 0.0) {
                    ihi = ilo - 1;
                } else {
                    const double rx = sqrt(rem) / A.dx + 0.5;
                    const int a = (int)ceil(ri - rx), z = (int)floor(ri + rx);
                    ilo = a > imin ? a : imin;
                    ihi = z < imax ? z : imax;
                }
                if (ilo <= ihi) {
                    const int rowbase = (j - 1) * A.nx;
                    const int lo = rowbase + ilo - 1, hi = rowbase + ihi - 1;
                    const int c0 = lo > 0 ? cc[lo - 1] : 0;
                    beg = bs + c0;
                    len = cc[hi] - c0;
                }
            }
            // the rows that hold candidates, 64 of one row at a time; the next chunk's
            // loads are on their way while one is tested.  Where that would leave the chunks
            // less than half full (not kDense), all rows as one sequence, 64 of it at a time,
            // each lane looking up its candidate's row among the sums of the lengths.
            int ntot = 0;
            bool packed = false;
            if constexpr (FORM != kDense) {
                ntot = __builtin_amdgcn_readlane(wave_scan(len), 63);
                const int nch = __builtin_amdgcn_readlane(wave_scan((len + 63) >> 6), 63);
                packed = 2 * ((ntot + 63) >> 6) <= nch;
            }
            for (int q0 = 0;; q0 += 64) {
                unsigned long long rows = __ballot(len > 0);
                int r = 0, rbeg = 0, rlen = 0, at = 0, np = -1;
                float4 nrec = make_float4(0.f, 0.f, 0.f, 0.f);
                auto row = [&]() {
                    r = __builtin_ctzll(rows);
                    rbeg = __builtin_amdgcn_readlane(beg, r);
                    rlen = __builtin_amdgcn_readlane(len, r);
                    at = 0;
                };
                auto fetch = [&]() {
                    np = at + lane < rlen ? rbeg + at + lane : -1;
                    if (np >= 0) nrec = A.brf[np];
                };
                if (FORM != kDense && packed && rows) {
                    const int pre = wave_scan(len), q = q0 + lane;
                    int k = 0;  // rows whose candidates all come before q
#pragma unroll
                    for (int d = 32; d > 0; d >>= 1)
                        if (__shfl(pre, k + d - 1, 64) <= q) k += d;
                    const int p0 = __shfl(beg - (pre - len), k, 64);
                    np = q < ntot ? p0 + q : -1;
                    if (np >= 0) nrec = A.brf[np];
                    r = __builtin_amdgcn_readfirstlane(k);
                    rows = 1;  // one chunk
                } else if (rows) {
                    row();
                    fetch();
                }
                do {
                    if (rows) {
                        if (at == 0 && S.m >= cap && (double)(j0 + r) - rj > 0.5) {
                            // rows from this one on lie beyond the point: an obs of
                            // row j has |rj_o - rj| > j - rj - 0.5, so
                            // nd > ((j - rj - 0.5) dy / sigma_h)^2 and its key
                            // err^2 / rho exceeds err2_min exp(nd / 2); once that
                            // bound (less a 1e-9 margin for rounding) reaches tau,
                            // which only falls, no later candidate can enter
                            const double g = ((double)(j0 + r) - rj - 0.5) * A.dy / A.sigma_h;
                            const double lb = e2min * exp(0.5 * g * g) * (1.0 - 1e-9);
                            if (lb >= __longlong_as_double((long long)S.tau)) {
                                fin = true;
                                rows = 0;
                            }
                        }
                    }
                    if (rows) {
                        const float4 cur = nrec;
                        const int p = np;
                        at += 64;
                        if (at >= rlen) {
                            rows &= rows - 1;
                            if (rows) row();
                        }
                        if (rows) fetch();
                        const float fx = fri - cur.x, fy = frj - cur.y, fz = cur.z - frz;
                        const float nd = __builtin_fmaf(fx * fx, cx,
                                                        __builtin_fmaf(fy * fy, cy, fz * fz * cv));
                        bool in = p >= 0 && !(nd > nd_out);
                        if (S.n < cap) {
                            if (in && !(nd < nd_in))
                                in = eval_rec(A, load_rec(p), p, ri, rj, rz).ok;
                        } else if (S.m >= cap) {
                            in = in && !(__builtin_fmaf(0.72134752f, nd, cur.w) > l2tau);
                        }
                        wc_push(W, S, in, p, cap, lane);
                    }
                    const unsigned long long tau0 = S.tau;
                    wc_service<FORM == kSmallCap>(W, so, S, cap, lane, fin, eval);
                    if (S.tau != tau0)
                        // 0.73 em for nd's error, 1e-3 for the logarithms'
                        l2tau = (float)log2(__longlong_as_double((long long)S.tau)) + 0.73f * em +
                                1.0e-3f;
                } while (rows);
                if (FORM == kDense || !packed || fin || q0 + 64 >= ntot) break;
            }
            if (fin) break;
        }
        const int kept = S.n < cap ? S.n : cap;
        if (lane == 0) W.cnt[0] = (unsigned)kept;  // (the counts are spent)
        __syncthreads();
        int off = 0, tot = 0;
        for (int u = 0; u < NW; ++u) {
            const int k = (int)L[u].cnt[0];
            off += u < wv ? k : 0;
            tot += k;
        }
        const long obase = A.list_off[b] - A.list_base;  // relative to this chunk's list buffer
        const int* from = S.n < cap ? wc_fill_pos(W) : so;
        for (int sl = lane; sl < kept; sl += 64) {
            const int p = from[sl];
            A.loc_idx[obase + off + sl] = A.bo[p];
            A.loc_rho[obase + off + sl] = eval_rec(A, load_rec(p), p, ri, rj, rz).rho;
        }
        if (threadIdx.x == 0) {
            A.loc_off[b] = obase;
            A.loc_cnt[b] = tot;
        }
        __syncthreads();
    }
}

// The bucket-by-bucket copy of the sorted obs: per cell, its obs of each
// bucket (count), then each bucket's inclusive scan over cells, then the copy
// (every cell's obs in order, each to its bucket's next position).
__global__ void reg_bucket_count(const int* cellcum, const int* obkt, int ncell, int nbkt,
                                 int* bcnt)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    int n[LEKF_REG_NB] = {0, 0, 0, 0};
    const int beg = c > 0 ? cellcum[c - 1] : 0, end = cellcum[c];
    for (int i = beg; i < end; ++i) {
        const int t = obkt[i];
        if (t >= 0 && t < LEKF_REG_NB) ++n[t];
    }
    for (int t = 0; t < nbkt; ++t) bcnt[(size_t)t * ncell + c] = n[t];
}

__global__ void reg_bucket_scatter(const int* cellcum, const double* ori, const double* orj,
                                   const double* oz, const double* oerr, const int* obkt,
                                   int ncell, int nbkt, const int* bcc, double* brec,
                                   float4* brf, int* bo, unsigned long long* err2_min)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    int pos[LEKF_REG_NB] = {0, 0, 0, 0};
    int bs = 0;
    for (int t = 0; t < nbkt; ++t) {
        const int* cc = bcc + (size_t)t * ncell;
        pos[t] = bs + (c > 0 ? cc[c - 1] : 0);
        bs += cc[ncell - 1];
    }
    const int beg = c > 0 ? cellcum[c - 1] : 0, end = cellcum[c];
    unsigned long long e2[LEKF_REG_NB] = {~0ull, ~0ull, ~0ull, ~0ull};
    for (int i = beg; i < end; ++i) {
        const int t = obkt[i];
        if (t < 0 || t >= nbkt) continue;
        const int p = pos[t]++;
        double* r = brec + 4 * (size_t)p;
        r[0] = ori[i];
        r[1] = orj[i];
        r[2] = oz[i];
        r[3] = oerr[i];
        brf[p] = make_float4((float)ori[i], (float)orj[i], (float)oz[i],
                             (float)log2(rn_mul(oerr[i], oerr[i])));
        bo[p] = i;
        // err^2 >= 0: its bits order as the values do
        const unsigned long long b2 = (unsigned long long)__double_as_longlong(rn_mul(oerr[i], oerr[i]));
        for (int u = 0; u < LEKF_REG_NB; ++u)
            if (u == t && b2 < e2[u]) e2[u] = b2;
    }
    for (int u = 0; u < nbkt && u < LEKF_REG_NB; ++u)
        if (e2[u] != ~0ull) atomicMin(&err2_min[u], e2[u]);
}

// Nearest-first cap of the global grid's per-point lists: a list longer than
// the cap keeps the cap entries of largest rho (ties: the earlier list entry)
// in the reference's storage-slot order, by the cap of
// scale/letkf/letkf_tools.f90:1041-1156 with the key 2^63 - 1 - bits(rho)
// (rho > 0; a smaller key is a larger rho).  list_cap_wave: one wave per point
// (persistent), caps up to LEKF_CAP_LDS; list_cap: one workgroup per point.
__device__ __forceinline__ unsigned long long rho_key(double rho)
{
    return 0x7fffffffffffffffull - (unsigned long long)__double_as_longlong(rho);
}

template <bool SMALL>
__global__ __launch_bounds__(64) void list_cap_wave(ListCapArgs A)
{
    __shared__ WaveCap L;
    __shared__ int so[LEKF_CAP_LDS];
    const int lane = threadIdx.x;
    const long npt = (long)A.ncols * A.nlev;
    for (long pi = blockIdx.x; pi < npt; pi += gridDim.x) {
        const long b = (pi / A.ncols) * (long)A.nij + A.col_begin + pi % A.ncols;
        const long off = A.in_off[b];
        const int n = A.in_cnt[b];
        const long ob = b * (long)A.cap;
        const int* ii = A.in_idx + off;
        const double* ir = A.in_rho + off;
        int kept = n;
        if (n <= A.cap) {
            for (int i = lane; i < n; i += 64) {
                A.out_idx[ob + i] = ii[i];
                A.out_rho[ob + i] = ir[i];
            }
        } else {
            WcState S{0, 0, 0, ~0ull};
            double rn = lane < n ? ir[lane] : 0.0;
            for (int i0 = 0; i0 < n; i0 += 64) {
                const double rc = rn;
                const int i = i0 + lane;
                rn = i + 64 < n ? ir[i + 64] : 0.0;
                wc_push(L, S, i < n && rho_key(rc) < S.tau, i, A.cap, lane);
                wc_service<SMALL>(L, so, S, A.cap, lane, i0 + 64 >= n, [&](int p, bool& ok) {
                    ok = true;
                    return rho_key(ir[p]);
                });
            }
            kept = A.cap;
            for (int sl = lane; sl < kept; sl += 64) {
                const int i = so[sl];
                A.out_idx[ob + sl] = ii[i];
                A.out_rho[ob + sl] = ir[i];
            }
            wave_sync();
        }
        if (lane == 0) {
            A.out_off[b] = ob;
            A.out_cnt[b] = kept;
        }
    }
}

__global__ __launch_bounds__(kSelT) void list_cap(ListCapArgs A)
{
    __shared__ SelLds S;
    const int tid = threadIdx.x;
    CapGlobal G;
    G.key = A.g_key ? A.g_key + (size_t)blockIdx.x * 2 * A.cap : nullptr;
    G.pos = A.g_pos ? A.g_pos + (size_t)blockIdx.x * 2 * A.cap : nullptr;
    G.slot = A.g_slot ? A.g_slot + (size_t)blockIdx.x * 2 * A.cap : nullptr;
    const long npt = (long)A.ncols * A.nlev;
    for (long pi = blockIdx.x; pi < npt; pi += gridDim.x) {
        const long b = (pi / A.ncols) * (long)A.nij + A.col_begin + pi % A.ncols;
        const long off = A.in_off[b];
        const int n = A.in_cnt[b];
        const long ob = b * (long)A.cap;
        int kept = n;
        if (n <= A.cap) {
            for (int i = tid; i < n; i += kSelT) {
                A.out_idx[ob + i] = A.in_idx[off + i];
                A.out_rho[ob + i] = A.in_rho[off + i];
            }
        } else {
            const int* ii = A.in_idx + off;
            const double* ir = A.in_rho + off;
            kept = cap_stream(
                S, G, [&](int i) { return rho_key(ir[i]); },
                [&](int slot, int i) {
                    A.out_idx[ob + slot] = ii[i];
                    A.out_rho[ob + slot] = ir[i];
                },
                n, A.cap, tid);
        }
        if (tid == 0) {
            A.out_off[b] = ob;
            A.out_cnt[b] = kept;
        }
        __syncthreads();
    }
}

// per point: candidate count of the rectangle -> list capacity
__global__ void reg_capacity(RegionalArgs A, int* capn, int* maxcand)
{
    const long b = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long npt = (long)A.nx * A.ny * A.nlev;
    if (b >= npt) return;
    const int nij = A.nx * A.ny;
    const int ij = (int)(b % nij);
    const double ri = (double)(ij % A.nx + 1), rj = (double)(ij / A.nx + 1);
    int imin = (int)floor(ri - A.dlon_zero), imax = (int)ceil(ri + A.dlon_zero);
    int jmin = (int)floor(rj - A.dlat_zero), jmax = (int)ceil(rj + A.dlat_zero);
    if (imin < 1) imin = 1;
    if (imax > A.nx) imax = A.nx;
    if (jmin < 1) jmin = 1;
    if (jmax > A.ny) jmax = A.ny;
    long n = 0;
    for (int j = jmin; j <= jmax && imin <= imax; ++j) {
        const long rowbase = (long)(j - 1) * A.nx;
        const int beg = (imin > 1) ? A.cellcum[rowbase + imin - 2] : (rowbase > 0 ? A.cellcum[rowbase - 1] : 0);
        n += A.cellcum[rowbase + imax - 1] - beg;
    }
    atomicMax(maxcand, (int)n);
    if (A.nobs_max > 0) {
        const long c = (long)A.nobs_max * A.nbkt;
        n = n < c ? n : c;
    }
    capn[b] = (int)n;
}

// obs keys: cell (ceiling(ri-0.5), ceiling(rj-0.5)) clamped; qc-rejected obs sort last
__global__ void reg_keys(RegObsArgs A)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= A.nobs) return;
    unsigned long long key = ~0ull;
    if (!A.qc || A.qc[n] == A.qc_keep) {
        int i = (int)ceil(A.ri[n] - 0.5), j = (int)ceil(A.rj[n] - 0.5);
        i = i < 1 ? 1 : (i > A.nx ? A.nx : i);
        j = j < 1 ? 1 : (j > A.ny ? A.ny : j);
        const unsigned cell = (unsigned)((i - 1) + A.nx * (j - 1));
        key = ((unsigned long long)cell << 32) | (unsigned)n;
        atomicAdd(&A.cell_cnt[cell], 1);
    }
    A.keys[n] = key;
}

__global__ void reg_scatter(RegObsArgs A, int nbinned)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nbinned) return;
    const int n = (int)(A.keys[m] & 0xffffffffull);
    A.perm[m] = n;
    A.o_ri[m] = A.ri[n];
    A.o_rj[m] = A.rj[n];
    A.o_z[m] = A.z[n];
    A.o_err[m] = A.err[n];
    A.o_rdiag[m] = A.err[n] * A.err[n];
    A.o_dep[m] = A.dep[n];
    A.o_bkt[m] = A.bkt[n];
    for (int i = 0; i < A.ne; ++i) {
        const double v = A.hdxf[(size_t)n * A.h_so + (size_t)i * A.h_sm];
        A.o_hdxf[(size_t)m * A.ne + i] = v;
        if (A.o_hdxf32) A.o_hdxf32[(size_t)m * A.ne + i] = (float)v;
    }
}

__global__ __launch_bounds__(1024) void scan_inclusive_int(const int* in, int* out, int n)
{
    __shared__ int s[1024];
    int carry = 0;
    for (int base = 0; base < n; base += 1024) {
        const int i = base + threadIdx.x;
        const int v = i < n ? in[i] : 0;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const int t = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
            __syncthreads();
            s[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < n) out[i] = carry + s[threadIdx.x];
        const int tot = s[1023];
        __syncthreads();
        carry += tot;
    }
}

__global__ __launch_bounds__(1024) void scan_exclusive_long(const int* in, long* out, long n)
{
    __shared__ long s[1024];
    long carry = 0;
    for (long base = 0; base < n; base += 1024) {
        const long i = base + threadIdx.x;
        const long v = i < n ? in[i] : 0;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const long t = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
            __syncthreads();
            s[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < n) out[i] = carry + s[threadIdx.x] - v;
        const long tot = s[1023];
        __syncthreads();
        carry += tot;
    }
    if (threadIdx.x == 0) out[n] = carry;
}

}  // namespace

hipError_t lekf_reg_keys_launch(const RegObsArgs& A, hipStream_t st)
{
    if (A.nobs > 0)
        hipLaunchKernelGGL(reg_keys, dim3((A.nobs + 255) / 256), dim3(256), 0, st, A);
    return hipGetLastError();
}

hipError_t lekf_reg_scatter_launch(const RegObsArgs& A, int nbinned, int ncell, int* cellcum,
                                   hipStream_t st)
{
    if (nbinned > 0)
        hipLaunchKernelGGL(reg_scatter, dim3((nbinned + 255) / 256), dim3(256), 0, st, A, nbinned);
    hipLaunchKernelGGL(scan_inclusive_int, dim3(1), dim3(1024), 0, st, A.cell_cnt, cellcum, ncell);
    return hipGetLastError();
}

hipError_t lekf_reg_capacity_launch(const RegionalArgs& A, int* capn, long* cap_off, int* maxcand,
                                    hipStream_t st)
{
    const long npt = (long)A.nx * A.ny * A.nlev;
    hipLaunchKernelGGL(reg_capacity, dim3((unsigned)((npt + 255) / 256)), dim3(256), 0, st, A, capn,
                       maxcand);
    hipLaunchKernelGGL(scan_exclusive_long, dim3(1), dim3(1024), 0, st, capn, cap_off, npt);
    return hipGetLastError();
}

// workgroup slots of the persistent selection (LDS allows up to four per CU)
int lekf_reg_select_slots()
{
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    const int per = g_lekf_tune.sel_per_cu < 1 ? 1 : (g_lekf_tune.sel_per_cu > 4 ? 4 : g_lekf_tune.sel_per_cu);
    return per * (ncu > 0 ? ncu : 256);
}

int lekf_reg_select_slots_max()
{
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    return 4 * (ncu > 0 ? ncu : 256);
}

// a CU holds at most 16 waves of the fused selection (its LDS and registers)
long lekf_reg_wave_slots_max()
{
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    return 16L * (ncu > 0 ? ncu : 256);
}

// Workgroups of `lds` bytes that a CU holds: 160 KB in granules of 1280 bytes (the
// occupancy query counts bytes, and a persistent workgroup too many waits for a whole
// one to end, which nearly doubles the launch)
static constexpr int lds_fit(size_t lds) { return (int)(128 / ((lds + 1279) / 1280)); }

// Largest cap merged in blocks of 64.  96 x 48 x 7 points, 4000 stations, list_cap_wave at
// caps 10 / 40 / 64 / 100: 1.08 / 1.41 / 1.62 / 1.91 ms so, 1.34 / 1.53 / 1.63 / 1.75 in
// blocks of 224.
constexpr int kSmallCapMax = 64;

hipError_t lekf_list_cap_launch(const ListCapArgs& A, int nslots, hipStream_t st)
{
    const long npt = (long)A.ncols * A.nlev;
    if (npt <= 0) return hipSuccess;
    KTime kt("list_cap", st);
    if (A.cap <= LEKF_CAP_LDS) {
        // one wave per point: as many as the LDS lets a CU hold
        int dev = 0, ncu = 256, per_cu = 1;
        if (hipGetDevice(&dev) == hipSuccess)
            (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        const auto fn = A.cap <= kSmallCapMax ? list_cap_wave<true> : list_cap_wave<false>;
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 64, 0);
        per_cu = std::min(per_cu, lds_fit(sizeof(WaveCap) + sizeof(int) * LEKF_CAP_LDS));
        long g = (long)(per_cu > 0 ? per_cu : 1) * (ncu > 0 ? ncu : 256);
        if (g > npt) g = npt;
        hipLaunchKernelGGL(fn, dim3((unsigned)g), dim3(64), 0, st, A);
        return hipGetLastError();
    }
    const long g = npt < nslots ? npt : nslots;
    hipLaunchKernelGGL(list_cap, dim3((unsigned)g), dim3(kSelT), 0, st, A);
    return hipGetLastError();
}

template <int NW, int FORM>
static hipError_t launch_select_wave(const RegionalArgs& A, long npt, hipStream_t st)
{
    // as many workgroups as the LDS lets the CUs hold
    int dev = 0, ncu = 256, per_cu = 1;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (reg_select_wave<NW, FORM>), 64 * NW,
                                                       0);
    per_cu = std::min(per_cu, lds_fit(NW * sizeof(WaveCap)));
    long g = (long)(per_cu > 0 ? per_cu : 1) * (ncu > 0 ? ncu : 256);
    if (g * NW > A.wc_so_waves) g = A.wc_so_waves / NW;  // one slot map per wave
    if (g > npt) g = npt;
    if (g < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((reg_select_wave<NW, FORM>), dim3((unsigned)g), dim3(64 * NW), 0, st, A,
                       npt);
    return hipGetLastError();
}

// Rows of fewer candidates than this, on average over the grid and per bucket, share chunks
constexpr double kFewRow = 32.0;

// Which form of reg_select_wave: 64 x 64 x 10 points, two buckets, ms with kSmallCap /
// kFewRows / kDense at cap 10: 0.42 / 0.57 / 1.16 (3 candidates a row), 0.79 / 0.92 / 1.33 (15),
// 1.93 / 2.36 / 2.37 (150); at cap 100: 0.18 / 0.20 / 0.59, 1.05 / 0.97 / 1.40, 3.31 / 3.08 /
// 3.09; at cap 500: 0.18 / 0.20 / 0.59, 0.40 / 0.45 / 0.72, 6.60 / 4.73 / 4.67.  At 30
// candidates a row, cap 500, kFewRows 1.63 and kDense 1.79; at 60 they are alike.
template <int NW>
static hipError_t launch_select_form(const RegionalArgs& A, long npt, hipStream_t st)
{
    if (A.nobs_max <= kSmallCapMax) return launch_select_wave<NW, kSmallCap>(A, npt, st);
    const double row = (2.0 * std::sqrt(kNdMax) * A.sigma_h / A.dx + 1.0) * A.nbinned /
                       ((double)A.nbkt * A.nx * A.ny);
    return row < kFewRow ? launch_select_wave<NW, kFewRows>(A, npt, st)
                         : launch_select_wave<NW, kDense>(A, npt, st);
}

hipError_t lekf_reg_select_launch(const RegionalArgs& A, long npt, int nslots, hipStream_t st)
{
    if (npt <= 0) return hipSuccess;
    KTime kt("select", st);
    if (lekf_reg_select_fused(A.nobs_max) && A.bcc) {
        switch (A.nbkt) {
        case 1: return launch_select_form<1>(A, npt, st);
        case 2: return launch_select_form<2>(A, npt, st);
        case 3: return launch_select_form<3>(A, npt, st);
        case 4: return launch_select_form<4>(A, npt, st);
        default: return hipErrorInvalidValue;
        }
    }
    const long g = npt < nslots ? npt : nslots;
    hipLaunchKernelGGL(reg_select, dim3((unsigned)g), dim3(kSelT), 0, st, A, npt);
    return hipGetLastError();
}

hipError_t lekf_reg_buckets_launch(const RegObsArgs& A, int nbinned, const int* cellcum, int nbkt,
                                   int* bcnt, int* bcc, double* brec, float4* brf, int* bo,
                                   unsigned long long* err2_min, hipStream_t st)
{
    (void)nbinned;
    const int ncell = A.nx * A.ny;
    if (ncell <= 0 || nbkt < 1 || nbkt > LEKF_REG_NB) return hipErrorInvalidValue;
    const int nb = (ncell + 255) / 256;
    hipLaunchKernelGGL(reg_bucket_count, dim3(nb), dim3(256), 0, st, cellcum, A.o_bkt, ncell, nbkt,
                       bcnt);
    for (int t = 0; t < nbkt; ++t)
        hipLaunchKernelGGL(scan_inclusive_int, dim3(1), dim3(1024), 0, st, bcnt + (size_t)t * ncell,
                           bcc + (size_t)t * ncell, ncell);
    hipLaunchKernelGGL(reg_bucket_scatter, dim3(nb), dim3(256), 0, st, cellcum, A.o_ri, A.o_rj,
                       A.o_z, A.o_err, A.o_bkt, ncell, nbkt, bcc, brec, brf, bo, err2_min);
    return hipGetLastError();
}
