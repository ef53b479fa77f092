// Records in row form: the data pass for tracks whose equations each touch the parameters of one
// group only (the usual detector hit) and whose local fit has at most 5 parameters.
//
// At structure time such a record is laid out as one dense row per equation (value, error, local
// derivatives, derivatives of the group's parameters; the payload's own type), with a table of the
// groups it touches and the equations of each (k_rows_class, k_rows_fill).  A pass then needs no
// index words: one wavefront takes a record, one lane an equation (k_rows_pass).
//
// Matrix-building passes with group-block storage do not write the record's update (n(n+1)/2
// values for n parameters) but its factors.  With Gamma = sum_e w_e l_e l_e^T the update is
//     sum_e w_e g_e g_e^T - sum_ef g_e s_ef g_f^T,   s_ef = w_e w_f l_e^T Gamma^-1 l_f = q_e S q_f,
//     q_e = w_e |D|^-1/2 L^-1 l_e,  Gamma = L D L^T in the pivot order of the local fit, S = sgn D,
// so the q_e (k values for k local parameters) and g_e of two equations determine their
// contribution to the block of their groups.  The equations of a group are kept in units of two
// (128 bytes for FP32 records with 4 local parameters and 6 parameters in a group).
// k_rows_gather forms the products of all pairs of units that meet in a block while it sums them
// (k_rows_gather_diag: diagonal blocks, vector and counters, with w_e and w_e r_e from a side
// array).  Both sum in processing order, so passes repeat bit for bit.
//
// Why: for 18 hits of 6 parameters the update is 6,000 values (48 KB), the factors are 2.9 KB.
// Written and read once, the updates of 2,000,000 such tracks are 200 GB of HBM traffic.
//
// The arithmetic of the local fit is that of k_records (loopbf, src/pede.f90:3655-4229): sums over
// the equations in record order, sqminv's pivot order, the same chi^2 reductions.
#include "mpgpu_internal.h"
#include <hipcub/hipcub.hpp>
#include <float.h>
#include <algorithm>

namespace mpgpu {

#define WV 64
#define RWAVES 4                 // wavefronts (records in flight) per workgroup of the pass
#define MAXEQ 128                // equations per record: two per lane
#define MAXGRP 8                 // parameters of a group (fixed ones included)
#define MAXSEG 128               // groups, and units, per record
#define PERM_WINDOW 4096         // blocks whose order the gather may change
#define MAXSEQ 4                 // equations of one group in a record

__device__ __forceinline__ double rsum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WV);
    return v;
}

// ---------------------------------------------------------------------------------------------
// structure: which records have row form, and their rows
// ---------------------------------------------------------------------------------------------
// One wavefront per record.  cls[r] = 1 when every equation's labels lie in one group of at most
// MAXGRP parameters, each once, the local indices are within 1..5, each once, no group has more
// than MAXSEQ equations, and the counts fit.  n[0..3][r]: equations, groups, units, pairs of units.
__global__ __launch_bounds__(WV *RWAVES) void k_rows_class(int64_t nrec, const int64_t *rec_eq, const int64_t *eq_sl,
                                                           const uint32_t *eq_n, const int32_t *widx,
                                                           const int64_t *rec_gl, const int32_t *gl_tix,
                                                           const int32_t *band, RowGroups Q, uint8_t *cls, int32_t *n,
                                                           int32_t *maxes)
{
    __shared__ int32_t s_eg[RWAVES][MAXEQ];
    const int lane = threadIdx.x & (WV - 1);
    int32_t *eg = s_eg[threadIdx.x >> 6];
    int mx_eq = 0, mx_nl = 0, mx_g = 0;
    for (int64_t r = blockIdx.x * (int64_t)RWAVES + (threadIdx.x >> 6); r < nrec; r += (int64_t)gridDim.x * RWAVES) {
        const int64_t e0 = rec_eq[r], g0 = rec_gl[r];
        const int neq = (int)min(rec_eq[r + 1] - e0, (int64_t)(MAXEQ + 1)), ngl = (int)(rec_gl[r + 1] - g0);
        bool bad = neq > MAXEQ || (band && band[r] != 0);
        int nl_max = 0, gs_max = 0;
        if (!bad) {
            for (int i = lane; i < neq; i += WV) {
                const int64_t sl = eq_sl[e0 + i];
                const uint32_t en = eq_n[e0 + i];
                const int nl = en & 0xffff, ng = en >> 16;
                unsigned lm = 0;
                int tgi = -1;
                if (nl > 5) bad = true;
                else
                    for (int j = 1; j <= nl; j++) {
                        const int ij = widx[sl + j];
                        if (ij < 1 || ij > 5 || ((lm >> ij) & 1u)) { bad = true; break; }
                        lm |= 1u << ij;
                        nl_max = max(nl_max, ij);
                    }
                if (ng > MAXGRP) bad = true;
                else if (ng > 0) {
                    const int64_t sg = sl + nl + 1;
                    const int tg = Q.of[gl_tix[g0 + widx[sg + 1]]], t0 = Q.t0[tg], sz = Q.t0[tg + 1] - t0;
                    tgi = tg;
                    gs_max = max(gs_max, sz);
                    if (sz > MAXGRP) bad = true;
                    else {
                        unsigned gm = 0;
                        for (int j = 1; j <= ng; j++) {
                            const int d = gl_tix[g0 + widx[sg + j]] - t0;
                            if (d < 0 || d >= sz || ((gm >> d) & 1u)) { bad = true; break; }
                            gm |= 1u << d;
                        }
                    }
                }
                eg[i] = tgi;
            }
        }
        bad = __any(bad);
        for (int o = 32; o > 0; o >>= 1) {
            nl_max = max(nl_max, __shfl_xor(nl_max, o, WV));
            gs_max = max(gs_max, __shfl_xor(gs_max, o, WV));
        }
        wave_order();
        // groups of the record: runs of its (sorted) label list; a group has units when one of its
        // variables is in the list
        int nseg = 0, nu = 0;
        if (!bad) {
            int lasttg = -1;
            for (int b0 = 0; b0 < ngl; b0 += WV) {
                const int k = b0 + lane;
                const int t = k < ngl ? gl_tix[g0 + k] : -1;
                const int tg = t >= 0 ? Q.of[t] : -1;
                const int up = __shfl_up(tg, 1, WV);
                const bool first = tg >= 0 && tg != (lane > 0 ? up : lasttg);
                lasttg = __shfl(tg, min(WV, ngl - b0) - 1, WV);
                int cnt = 0, live = 0;
                if (first) {
                    for (int i = 0; i < neq; i++) cnt += eg[i] == tg;
                    for (int x = k; x < ngl && Q.of[gl_tix[g0 + x]] == tg; x++) live |= Q.var[gl_tix[g0 + x]] > 0;
                    if (cnt > MAXSEQ) bad = true;
                }
                nseg += __popcll(__ballot(first));
                int u = live ? (cnt + 1) / 2 : 0;
                for (int o = 32; o > 0; o >>= 1) u += __shfl_xor(u, o, WV);
                nu += u;
            }
            if (nseg > MAXSEG || nu > MAXSEG) bad = true;
            bad = __any(bad);
        }
        if (lane == 0) {
            cls[r] = bad ? 0 : 1;
            n[r] = bad ? 0 : neq;
            n[nrec + r] = bad ? 0 : nseg;
            n[2 * nrec + r] = bad ? 0 : nu;
            n[3 * nrec + r] = bad ? 0 : nu * (nu + 1) / 2;
        }
        if (!bad) {
            mx_eq = max(mx_eq, neq);
            mx_nl = max(mx_nl, nl_max);
            mx_g = max(mx_g, gs_max);
        }
        wave_order();
    }
    if (lane == 0) {
        atomicMax(&maxes[0], mx_eq);
        atomicMax(&maxes[1], mx_nl);
        atomicMax(&maxes[2], mx_g);
    }
}

// counts of the records in processing order (one array per count, an extra zero at the end)
__global__ void k_rows_counts(int64_t nq, int64_t nrec, const int64_t *order, const int32_t *n, int64_t *c)
{
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q <= nq; q += (int64_t)gridDim.x * blockDim.x)
        for (int k = 0; k < 4; k++) c[k * (nq + 1) + q] = q < nq ? n[k * nrec + order[q]] : 0;
}

// columns of a row: value, error, KP local derivatives, GP derivatives of the group's parameters
// (the variable ones first)
template <typename T, int KP, int GP> struct RowLayout {
    static constexpr int V = 16 / (int)sizeof(T);                   // values per 16 bytes
    static constexpr int RS = (2 + KP + GP + V - 1) / V * V;        // row stride
};
// A unit in pieces of 16 bytes: q of its two equations (NQ pieces each), then the two halves of the
// group derivatives (NH pieces each: HM values of the first equation, HM of the second, and the
// signs S, bit k: D_k < 0).  Four lanes load a unit in whole lines, one piece each at a time, and
// exchange pieces (k_rows_gather).
template <typename T, int KP, int GP> struct UnitLayout {
    static constexpr int HM = GP / 2;
    static constexpr int NQ = KP / 2;
    static constexpr int SG = 2 * HM * (int)sizeof(T);              // signs, byte offset in a half
    static constexpr int NH = (SG + 4 + 15) / 16;
    static constexpr int NP = 2 * (NQ + NH);
    static constexpr int BYTES = 16 * NP;
    static __host__ __device__ constexpr int q(int e) { return 16 * NQ * e; }
    static __host__ __device__ constexpr int h(int x) { return 16 * (2 * NQ + NH * x); }
};

// One wavefront per record: its header, rows, group table, the equations of each group and the
// place of each equation in the record's units (2 unit + half; bit 15: the other half is empty;
// 0xffff: no variable parameters).
template <typename T, int KP, int GP>
__global__ __launch_bounds__(WV *RWAVES) void k_rows_fill(int64_t nq, const int64_t *order, const int64_t *c, const T *val,
                                                          const int64_t *rec_eq, const int64_t *eq_sl,
                                                          const uint32_t *eq_n, const int32_t *widx,
                                                          const int64_t *rec_gl, const int32_t *gl_tix, RowGroups Q,
                                                          RowHdr *hdr, T *rows, int32_t *eq_t0, uint16_t *eq_pos,
                                                          uint16_t *seq, int4 *seg)
{
    constexpr int RS = RowLayout<T, KP, GP>::RS;
    __shared__ int32_t s_tg[RWAVES][MAXSEG], s_live[RWAVES][MAXSEG];
    __shared__ uint8_t s_es[RWAVES][MAXEQ];
    const int lane = threadIdx.x & (WV - 1), wv = threadIdx.x >> 6;
    int32_t *tgl = s_tg[wv], *live = s_live[wv];
    uint8_t *es = s_es[wv];
    for (int64_t q = blockIdx.x * (int64_t)RWAVES + wv; q < nq; q += (int64_t)gridDim.x * RWAVES) {
        const int64_t r = order[q], e0 = rec_eq[r], g0 = rec_gl[r];
        const int neq = (int)(rec_eq[r + 1] - e0), ngl = (int)(rec_gl[r + 1] - g0);
        const int64_t row0 = c[q], seg0 = c[(nq + 1) + q], unit0 = c[2 * (nq + 1) + q];
        int nseg = 0, lasttg = -1;
        for (int b0 = 0; b0 < ngl; b0 += WV) {
            const int k = b0 + lane;
            const int t = k < ngl ? gl_tix[g0 + k] : -1;
            const int tg = t >= 0 ? Q.of[t] : -1;
            const int up = __shfl_up(tg, 1, WV);
            const bool first = tg >= 0 && tg != (lane > 0 ? up : lasttg);
            lasttg = __shfl(tg, min(WV, ngl - b0) - 1, WV);
            const unsigned long long m = __ballot(first);
            if (first) {
                const int p = nseg + __popcll(m & ((1ull << lane) - 1ull));
                int lv = 0;
                for (int x = k; x < ngl && Q.of[gl_tix[g0 + x]] == tg; x++) lv |= Q.var[gl_tix[g0 + x]] > 0;
                tgl[p] = tg;
                live[p] = lv;
            }
            nseg += __popcll(m);
        }
        wave_order();
        int nalc = 0;
        for (int i = lane; i < neq; i += WV) {
            const int64_t sl = eq_sl[e0 + i];
            const uint32_t en = eq_n[e0 + i];
            const int nl = en & 0xffff, ng = en >> 16;
            const int64_t sg = sl + nl + 1;
            T *row = rows + (row0 + i) * RS;
            for (int k = 0; k < RS; k++) row[k] = (T)0;
            row[0] = val[sl];
            row[1] = val[sg];
            for (int j = 1; j <= nl; j++) {
                const int ij = widx[sl + j];
                row[1 + ij] = val[sl + j];
                nalc = max(nalc, ij);
            }
            int t0 = -1, sgi = 255;
            if (ng > 0) {
                const int tg = Q.of[gl_tix[g0 + widx[sg + 1]]];
                t0 = Q.t0[tg];
                for (int j = 1; j <= ng; j++) row[2 + KP + Q.col[gl_tix[g0 + widx[sg + j]]]] = val[sg + j];
                int lo = 0, hi = nseg - 1;             // the group's place in the (ascending) table
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (tgl[mid] < tg) lo = mid + 1;
                    else hi = mid;
                }
                sgi = lo;
            }
            eq_t0[row0 + i] = t0;
            es[i] = (uint8_t)sgi;
        }
        for (int o = 32; o > 0; o >>= 1) nalc = max(nalc, __shfl_xor(nalc, o, WV));
        wave_order();
        // equations of each group, ascending, and their places in the units
        int before = 0, ubefore = 0;
        for (int b0 = 0; b0 < nseg; b0 += WV) {
            const int k = b0 + lane;
            int cnt = 0;
            if (k < nseg)
                for (int i = 0; i < neq; i++) cnt += es[i] == k;
            const int un = k < nseg && live[k] ? (cnt + 1) / 2 : 0;
            int x = cnt, y = un;
            for (int d = 1; d < WV; d <<= 1) {
                const int a = __shfl_up(x, d, WV), b = __shfl_up(y, d, WV);
                if (lane >= d) { x += a; y += b; }
            }
            const int start = before + x - cnt, ustart = ubefore + y - un;
            if (k < nseg) {
                int p = 0;
                for (int i = 0; i < neq; i++)
                    if (es[i] == k) {
                        seq[row0 + start + p] = (uint16_t)i;
                        const bool alone = (p & 1) == 0 && p == cnt - 1;
                        eq_pos[row0 + i] = (uint16_t)(un > 0 ? (2 * ustart + p) | (alone ? 0x8000 : 0) : 0xffff);
                        p++;
                    }
                const int tg = tgl[k];
                seg[seg0 + k] = make_int4(Q.v0[tg], start | (cnt << 16), live[k] ? __popc(Q.mask[tg]) : 0, ustart | (un << 16));
            }
            before += __shfl(x, WV - 1, WV);
            ubefore += __shfl(y, WV - 1, WV);
        }
        for (int i = lane; i < neq; i += WV)
            if (es[i] == 255) eq_pos[row0 + i] = 0xffff;
        if (lane == 0) {
            RowHdr h;
            h.row0 = row0;
            h.seg0 = seg0;
            h.unit0 = unit0;
            h.rec = r;
            h.neq = neq;
            h.nseg = nseg;
            h.nalc = nalc;
            h.nunit = ubefore;
            hdr[q] = h;
        }
        wave_order();
    }
}

// (block, units) of every pair of units of the records [q0, q1); units relative to the batch
__global__ __launch_bounds__(WV *RWAVES) void k_rows_incidence(int64_t q0, int64_t q1, const RowHdr *hdr, const int4 *seg,
                                                               const int32_t *group_of, const uint32_t *bits,
                                                               const int64_t *wrank, const int64_t *pr0, int64_t ub,
                                                               uint32_t *key, uint2 *val)
{
    __shared__ int32_t s_g[RWAVES][MAXSEG];
    const int lane = threadIdx.x & (WV - 1), wv = threadIdx.x >> 6;
    int32_t *ug = s_g[wv];
    for (int64_t q = q0 + blockIdx.x * (int64_t)RWAVES + wv; q < q1; q += (int64_t)gridDim.x * RWAVES) {
        const RowHdr h = hdr[q];
        for (int k = lane; k < h.nseg; k += WV) {
            const int4 d = seg[h.seg0 + k];
            const int u0 = d.w & 0xffff, un = d.w >> 16;
            if (un > 0) {
                const int g = group_of[d.x];
                for (int u = 0; u < un; u++) ug[u0 + u] = g;
            }
        }
        wave_order();
        const int64_t out = pr0[q] - pr0[q0];
        const int np = h.nunit * (h.nunit + 1) / 2;
        const uint32_t base = (uint32_t)(h.unit0 - ub);
        for (int t = lane; t < np; t += WV) {
            int a = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
            while (a * (a + 1) / 2 > t) a--;
            while ((a + 1) * (a + 2) / 2 <= t) a++;
            const int b = t - a * (a + 1) / 2;
            const int64_t o = (int64_t)ug[a] * (ug[a] + 1) / 2 + ug[b];
            key[out + t] = (uint32_t)(wrank[o >> 5] + __popc(bits[o >> 5] & ((1u << (o & 31)) - 1u)));
            val[out + t] = make_uint2(base + a, base + b);
        }
        wave_order();
    }
}

// first position of every key (sorted), keys 0 .. nk: a search per key, since a thread that filled a
// gap between two keys took as long as the gap (few records in row form, 200,000 blocks: 45 ms)
__global__ void k_rows_ptr(int64_t n, const uint32_t *key, int64_t nk, uint32_t *ptr)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k <= nk; k += (int64_t)gridDim.x * blockDim.x) {
        int64_t lo = 0, hi = n;                  // keys below lo are < k, from hi on >= k
        while (lo < hi) {
            const int64_t mid = (lo + hi) / 2;
            if ((int64_t)key[mid] < k) lo = mid + 1;
            else hi = mid;
        }
        ptr[k] = (uint32_t)lo;
    }
}

// Slots that share a block in the gather, by the length of its list: with one slot a list of 32
// pairs takes 32 steps, longer ones are split so that no wavefront runs much longer than the rest.
__device__ __forceinline__ int len_class(uint32_t n) { return n >= 128u ? 0 : n >= 32u ? 1 : 2; }

// sort key of a block: its class (3: diagonal or empty), its window of neighbouring blocks, then
// descending list length
__global__ void k_rows_len(int64_t nb, const uint32_t *ptr, const int32_t *brg, const int32_t *bcol, uint64_t *key,
                           uint32_t *val, unsigned long long *ncls)
{
    __shared__ unsigned s_n[4];
    if (threadIdx.x < 4) s_n[threadIdx.x] = 0u;
    __syncthreads();
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nb; k += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t n = ptr[k + 1] - ptr[k];
        const int c = n == 0 || brg[k] == bcol[k] ? 3 : len_class(n);
        key[k] = ((uint64_t)c << 36) | ((uint64_t)(k / PERM_WINDOW) << 12) | (uint64_t)(4095u - min(n, 4095u));
        val[k] = (uint32_t)k;
        atomicAdd(&s_n[c], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 3 && s_n[threadIdx.x]) atomicAdd(&ncls[threadIdx.x], (unsigned long long)s_n[threadIdx.x]);
}

// ---------------------------------------------------------------------------------------------
// the pass
// ---------------------------------------------------------------------------------------------
// sqminv (src/mpnum.f90:97-213) for N <= 5 parameters held one packed element per lane (lanes
// 0 .. N(N+1)/2), the right-hand side in the next N lanes: pivots in the reference's order among
// the nalc parameters in use, elimination by lane shuffles.  The result (inverse, solution) goes
// to cb[0 .. NPK) and cb[NPK .. NPK+N); returns the rank.  st[step]: the step's pivot parameter,
// pivot, and the multipliers of the parameters not yet eliminated (zero for the others).
template <int N> struct GjStep { double pivot, mu[N]; int k, pad; };
template <int N>
__device__ __forceinline__ int rows_gj(double acc, int nalc, int lane, int J, int K, double *cb, GjStep<N> *st)
{
    constexpr int NPK = N * (N + 1) / 2;
    const double eps = 16.0 * DBL_EPSILON;
    auto pk = [](int i, int j) { return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i; };
    double cv = lane < NPK ? acc : 0.0;
    double bv = __shfl(acc, min(NPK + lane, WV - 1), WV);     // lane l < N: right-hand side l
    const int L1 = lane < N ? lane : 0;
    double dg[N];
#pragma unroll
    for (int j = 0; j < N; j++) dg[j] = eps * fabs(wave_lane(cv, j * (j + 1) / 2 + j));
    unsigned rem = (1u << nalc) - 1u;
    int nrank = 0;
    for (int step = 0; step < nalc; step++) {
        int k = -1;
        double vkk = 0.0;
#pragma unroll
        for (int j = 0; j < N; j++) {
            const double vjj = wave_lane(cv, j * (j + 1) / 2 + j);
            if (((rem >> j) & 1u) && fabs(vjj) > fmax(fabs(vkk), dg[j])) { vkk = vjj; k = j; }
        }
        k = __builtin_amdgcn_readfirstlane(k);
        if (k < 0) {
            // no acceptable pivot left: the remaining rows and columns are set to zero
            if (lane < NPK && ((rem >> J) & 1u) && ((rem >> K) & 1u)) cv = 0.0;
            if (lane < N && ((rem >> lane) & 1u)) bv = 0.0;
            break;
        }
        rem &= ~(1u << k);
        nrank++;
        const double vinv = 1.0 / vkk;
        const double coJ = __shfl(cv, pk(J, k), WV);
        const double coK = __shfl(cv, pk(K, k), WV);
        const double coL = __shfl(cv, pk(L1, k), WV);
        const double bk = wave_lane(bv, k) * vinv;
        if (lane < N) st[step].mu[lane] = ((rem >> lane) & 1u) ? coL * vinv : 0.0;
        if (lane == 0) { st[step].pivot = vkk; st[step].k = k; }
        double nv;
        if (J == k && K == k) nv = -vinv;
        else if (J == k) nv = vinv * coK;
        else if (K == k) nv = vinv * coJ;
        else nv = cv - (vinv * coK) * coJ;
        if (lane < NPK) cv = nv;
        if (lane < N) bv = (L1 == k) ? bk : bv - bk * coL;
    }
    if (lane < NPK) cb[lane] = -cv;
    if (lane < N) cb[NPK + lane] = bv;
    return nrank;
}


// LDS of one wavefront (bytes): weights and products [mq], the local inverse and solution, the
// elimination steps, local derivatives and (without BUILD) group derivatives of the equations
template <typename T, int KP, int GP> __host__ __device__ constexpr int rows_lds(int mq, bool build)
{
    return (2 * mq + 32 + 48) * 8 + (mq * (KP + (build ? 0 : GP)) * (int)sizeof(T) + 15) / 16 * 16;
}

// One wavefront per record, no workgroup barriers.  BUILD: write the record's units; otherwise add
// to the vector and the counters.
template <typename T, int KP, int GP, bool BUILD>
__global__ __launch_bounds__(WV *RWAVES) __attribute__((amdgpu_waves_per_eu(4))) void k_rows_pass(RowDev R, DevModel M, PassOpts o, RecOut out, int64_t q0,
                                                          int64_t q1, int mq)
{
    constexpr int N = KP == 6 ? 5 : KP;
    constexpr int NPK = N * (N + 1) / 2, NE = NPK + N;
    constexpr int RS = RowLayout<T, KP, GP>::RS;
    constexpr int VL = WV / GP * GP;            // lanes of the parameter stage: whole groups
    typedef UnitLayout<T, KP, GP> UL;
    extern __shared__ __align__(16) double lds[];
    const int lane = threadIdx.x & (WV - 1), wv = threadIdx.x >> 6;
    const double chuber = 1.345, cauchy = 2.3849;
    double *w = (double *)((char *)lds + (size_t)wv * rows_lds<T, KP, GP>(mq, BUILD));   // weights
    double *wr = w + mq;                        // residuals, later weight x residual
    double *cb = wr + mq;                       // local inverse, then the solution
    GjStep<N> *st = (GjStep<N> *)(cb + 32);     // elimination steps
    T *Ls = (T *)(cb + 32 + 48);                // local derivatives
    T *gs = Ls + mq * KP;                       // group derivatives
    // element of the local normal equations summed by this lane
    int J = 0, K = 0;
    if (lane < NPK) {
        while ((J + 1) * (J + 2) / 2 <= lane) J++;
        K = lane - J * (J + 1) / 2;
    } else if (lane < NE) {
        J = lane - NPK;
    }
    const bool rhs = lane >= NPK;
    const bool robust = o.nloopn != 1 && o.lhuber != 0;
    const bool frac = o.lhuber > 1 && o.dwcut != 0.0f;     // down-weighted fraction cut in force
    const int nter = robust ? o.lhuber : 1;
    const T *rows = (const T *)R.rows;

    for (int64_t q = q0 + blockIdx.x * (int64_t)RWAVES + wv; q < q1; q += (int64_t)gridDim.x * RWAVES) {
        const RowHdr h = R.hdr[__builtin_amdgcn_readfirstlane((int)(q - q0)) + q0];
        const int neq = h.neq, nalc = h.nalc;
        double r[2], s[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            r[c] = 0.0;
            s[c] = 1.0;
            const int i = lane + WV * c;
            if (c == 1 && neq <= WV) break;
            if (i >= neq) continue;
            const T *row = rows + (h.row0 + i) * RS;
            T v[RS];
#pragma unroll
            for (int k = 0; k < RS; k++) v[k] = row[k];
            const int t0 = R.eq_t0[h.row0 + i];
            double rm = (double)v[0];
            double re = (double)v[1];
            if (t0 >= 0) {
#pragma unroll
                for (int j = 0; j < GP; j++) {
                    const double g = (double)v[2 + KP + j];
                    const int t = min(t0 + j, R.ntot - 1);
                    const double p = M.par[R.ptix ? R.ptix[t] : t];
                    if (g != 0.0) rm = rm - g * p;
                }
            }
            // 'scaleerrors' (prepareRecords, src/mppar.f90:312-316)
            re = re * (t0 >= 0 ? o.esc[0] : o.esc[1]);
#pragma unroll
            for (int k = 0; k < KP; k++) Ls[i * KP + k] = v[2 + k];
            if (!BUILD) {
#pragma unroll
                for (int j = 0; j < GP; j++) gs[i * GP + j] = v[2 + KP + j];
            }
            wr[i] = rm;
            r[c] = rm;
            s[c] = re;
        }
        // ---- local fit (src/pede.f90:3759-4094) ----
        int status = nalc > 0 ? 0 : 7, nrank = 0, ndf = 0;     // 7: no local parameters
        double summ = 0.0;
        float resing = 0.0f;
        double fit[2] = {0.0, 0.0}, wt[2] = {0.0, 0.0};
        for (int iter = 1; iter <= nter && status == 0; iter++) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int i = lane + WV * c;
                if (i >= neq) continue;
                double wght = 1.0 / (s[c] * s[c]);
                if (robust && iter != 1) {
                    const double resid = r[c] - fit[c];
                    if (iter <= 3) {
                        if (fabs(resid) > chuber * s[c]) wght = wght * chuber * s[c] / fabs(resid);
                    } else {
                        const double t = resid / s[c] / cauchy;
                        wght = wght / (1.0 + t * t);
                    }
                }
                wt[c] = wght;
                w[i] = wght;
            }
            wave_order();
            double acc = 0.0;
            if (lane < NE) {
                // equations in order; the products are rounded before they are added, as the
                // reference's are
#pragma clang fp contract(off)
                int i = 0;
                for (; i + 4 <= neq; i += 4) {
                    double t[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const double a = (double)Ls[(i + u) * KP + J];
                        const double x = rhs ? wr[i + u] : a;
                        const double y = rhs ? a : (double)Ls[(i + u) * KP + K];
                        t[u] = w[i + u] * x * y;
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) acc = acc + t[u];
                }
                for (; i < neq; i++) {
                    const double a = (double)Ls[i * KP + J];
                    const double x = rhs ? wr[i] : a;
                    const double y = rhs ? a : (double)Ls[i * KP + K];
                    acc = acc + w[i] * x * y;
                }
            }
            nrank = rows_gj<N>(acc, nalc, lane, J, K, cb, st);
            wave_order();
            double b[N];
#pragma unroll
            for (int k = 0; k < N; k++) b[k] = cb[NPK + k];
            bool nan = false;
#pragma unroll
            for (int k = 0; k < N; k++)
                if (k < nalc && !(b[k] <= 0.0) && !(b[k] > 0.0)) nan = true;
            // residuals and chi^2 (3919-4035)
            double s_chi = 0.0, s_wt = 0.0;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int i = lane + WV * c;
                if (i >= neq) continue;
                double f = 0.0;
#pragma unroll
                for (int k = 0; k < N; k++) f = f + (double)Ls[i * KP + k] * b[k];
                fit[c] = f;
                const double rmeas = r[c] - f;
                double wght = 1.0 / (s[c] * s[c]);
                double dchi2 = wght * rmeas * rmeas;
                if (robust || frac) {
                    double fac = wght;
                    if (robust && iter != 1) {
                        if (iter <= 3) {
                            if (fabs(rmeas) > chuber * s[c]) {
                                fac = wght * chuber * s[c] / fabs(rmeas);
                                dchi2 = 2.0 * chuber * (fabs(rmeas) / s[c] - 0.5 * chuber);
                            }
                        } else {
                            const double t = rmeas / s[c] / cauchy;
                            fac = wght / (1.0 + t * t);
                            dchi2 = log(1.0 + t * t) * cauchy * cauchy;
                        }
                    }
                    const double down = 1.0 / sqrt(fac);
                    s_wt += s[c] / down;
                }
                s_chi += dchi2;
            }
            summ = rsum(s_chi);
            ndf = neq - nrank;
            if (frac) {
                const double suwt = rsum(s_wt);
                resing = ((float)neq - (float)suwt) / (float)neq;
            }
            if (nan) { status = 1; break; }
            if (nrank != nalc) { status = 2; break; }
            if (ndf <= 0) { status = 4; break; }
        }
        double chi_add = 0.0;
        int ndf_add = 0;
        if (status == 0) {
            // chi^2 cuts with REAL(4) thresholds (4106-4131)
            const float chichi = three_sigma_chi2(ndf);
            if (o.chicut >= 0.0f) {
                if (summ > (double)(o.chhuge * chichi)) status = 5;
                else if (o.chicut > 0.0f) {
                    const float chlimt = o.chicut * chichi;
                    if (summ > (double)chlimt) { status = 6; chi_add = (double)chlimt; ndf_add = ndf; }
                }
            }
            if (status == 0 && frac && resing > o.dwcut) {
                status = 6;
                chi_add = summ;
                ndf_add = ndf;
            }
        }
        status = __builtin_amdgcn_readfirstlane(status);
        char *U = BUILD ? (char *)R.unit + (h.unit0 - R.ub) * UL::BYTES : nullptr;
        double *S = BUILD ? R.side + (h.unit0 - R.ub) * 4 : nullptr;
        if (status != 0) {
            if (lane == 0) { out.status[h.rec] = (int8_t)status; out.chi2[h.rec] = chi_add; out.ndf[h.rec] = ndf_add; }
            if (BUILD) {
                // a rejected record contributes nothing
                for (int t = lane; t < h.nunit * (UL::BYTES / 16); t += WV) ((double2 *)U)[t] = make_double2(0.0, 0.0);
                for (int t = lane; t < h.nunit * 4; t += WV) S[t] = 0.0;
            }
            continue;
        }
        // chi^2 of the accepted fit and the weights of the global update (4162-4183)
        double s_chi = 0.0;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int i = lane + WV * c;
            if (i >= neq) continue;
            const double rmeas = r[c] - fit[c];
            double wght = 1.0 / (s[c] * s[c]);
            double dchi2 = wght * rmeas * rmeas;
            if (robust) {
                const double resid = fabs(rmeas);
                if (nter <= 3) {
                    if (resid > chuber * s[c]) dchi2 = 2.0 * chuber * (resid / s[c] - 0.5 * chuber);
                } else {
                    const double t = resid / s[c] / cauchy;
                    dchi2 = log(1.0 + t * t) * cauchy * cauchy;
                }
                wght = wt[c];
            }
            s_chi += dchi2;
            if (!BUILD) {
                w[i] = wght;
                wr[i] = wght * rmeas;
                continue;
            }
            // q = w |D|^-1/2 L^-1 l: forward elimination of l in the pivot order of the local fit
            const unsigned pos = R.eq_pos[h.row0 + i];
            if (pos == 0xffffu) continue;
            double l[N], qv[KP];
            int sg = 0;
#pragma unroll
            for (int k = 0; k < N; k++) l[k] = (double)Ls[i * KP + k];
#pragma unroll
            for (int k = 0; k < KP; k++) qv[k] = 0.0;
#pragma unroll
            for (int t = 0; t < N; t++) {
                if (t >= nalc) break;
                const int k = st[t].k;
                const double p = st[t].pivot;
                double y = 0.0;
#pragma unroll
                for (int m = 0; m < N; m++)
                    if (m == k) y = l[m];
                qv[t] = wght * y / sqrt(fabs(p));
                if (p < 0.0) sg |= 1 << t;
#pragma unroll
                for (int m = 0; m < N; m++) l[m] = l[m] - st[t].mu[m] * y;
            }
            const int un = (int)((pos & 0x7fffu) >> 1), half = (int)(pos & 1u);
            char *u = U + (int64_t)un * UL::BYTES;
            double *uq = (double *)(u + UL::q(half));
#pragma unroll
            for (int k = 0; k < KP; k += 2) *(double2 *)&uq[k] = make_double2(qv[k], qv[k + 1]);
            const T *row = rows + (h.row0 + i) * RS + 2 + KP;
#pragma unroll
            for (int x = 0; x < 2; x++) {
                T *ug = (T *)(u + UL::h(x)) + half * UL::HM;
#pragma unroll
                for (int j = 0; j < UL::HM; j++) ug[j] = row[x * UL::HM + j];
                if (half == 0) *(int *)(u + UL::h(x) + UL::SG) = sg;
            }
            S[4 * un + half] = wght;
            S[4 * un + 2 + half] = wght * rmeas;
            if (pos & 0x8000u) {
                // no second equation in this unit
                double *u1 = (double *)(u + UL::q(1));
#pragma unroll
                for (int k = 0; k < KP; k += 2) *(double2 *)&u1[k] = make_double2(0.0, 0.0);
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int j = 0; j < UL::HM; j++) ((T *)(u + UL::h(x)))[UL::HM + j] = (T)0;
                S[4 * un + 1] = 0.0;
                S[4 * un + 3] = 0.0;
            }
        }
        summ = rsum(s_chi);
        if (lane == 0) { out.status[h.rec] = 0; out.chi2[h.rec] = summ; out.ndf[h.rec] = ndf; }
        wave_order();
        if (BUILD) continue;
        // ---- vector and counters (4184-4186): one lane per parameter of the record's groups ----
        for (int base = 0; base < h.nseg * GP; base += VL) {
            const int u = base + lane, sgi = u / GP, j = u - sgi * GP;
            const bool in = lane < VL && sgi < h.nseg;
            const int4 d = in ? R.seg[h.seg0 + sgi] : make_int4(0, 0, 0, 0);
            if (j >= d.z) continue;
            const int es = d.y & 0xffff, en = d.y >> 16;
            double v = 0.0;
            int cnt = 0;
            for (int x = 0; x < en; x++) {
                const int i = R.seq[h.row0 + es + x];
                const double gj = (double)gs[i * GP + j];
                v = v + wr[i] * gj;
                cnt += gj != 0.0;
            }
            atomicAdd(&M.vec[d.x + j - 1], v);
            atomicAdd(&M.cnt[d.x + j - 1], (unsigned long long)cnt);
        }
        wave_order();
    }
}

// ---------------------------------------------------------------------------------------------
// gather
// ---------------------------------------------------------------------------------------------
// consecutive workgroups go to different XCDs; each XCD takes runs of `run` neighbouring ones, so
// that the blocks of a block row, which read the same records, share an L2
__device__ __forceinline__ int64_t xcd_run(int64_t id, int64_t n, int run)
{
    const int64_t full = n / (8 * run) * (8 * run);
    if (id >= full) return id;
    const int64_t x = id & 7, k = id >> 3;
    return ((k / run) * 8 + x) * run + k % run;
}

// value of another lane of the same four (quad permutation)
template <int P> __device__ __forceinline__ double quad(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), P, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), P, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int R> __device__ __forceinline__ double row_ror(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + R, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + R, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// one dword of lane A (even half) / lane B (odd half) of the four; HI: the half is bit 1 of the
// lane, else bit 0.  Pieces 0, 1, ... lie in loads 0, 0, 0, 0, 1, ... of lanes 0, 1, 2, 3, 0, ...
template <int PERM> __device__ __forceinline__ int quad_i(int v) { return __builtin_amdgcn_mov_dpp(v, PERM, 0xf, 0xf, true); }
template <int A, int B, bool HI, int NI> __device__ __forceinline__ int4 piece(const int4 (&w)[NI], bool odd)
{
    constexpr int a = A & 3, b = B & 3;
    if constexpr (A / 4 == B / 4) {
        constexpr int P = HI ? a | a << 2 | b << 4 | b << 6 : a | b << 2 | a << 4 | b << 6;
        const int4 v = w[A / 4];
        return make_int4(quad_i<P>(v.x), quad_i<P>(v.y), quad_i<P>(v.z), quad_i<P>(v.w));
    } else {
        constexpr int P = a * 0x55, Q = b * 0x55;
        const int4 v = w[A / 4], u = w[B / 4];
        // both exchanges by all lanes, then the choice
        const int4 x = make_int4(quad_i<P>(v.x), quad_i<P>(v.y), quad_i<P>(v.z), quad_i<P>(v.w));
        const int4 y = make_int4(quad_i<Q>(u.x), quad_i<Q>(u.y), quad_i<Q>(u.z), quad_i<Q>(u.w));
        return odd ? y : x;
    }
}
// pieces BASE.. (even half) or BASE + N.. (odd half)
template <int BASE, int N, bool HI, int NI, int I = 0>
__device__ __forceinline__ void pieces(const int4 (&w)[NI], bool odd, int4 *out)
{
    if constexpr (I < N) {
        out[I] = piece<BASE + I, BASE + N + I, HI>(w, odd);
        pieces<BASE, N, HI, NI, I + 1>(w, odd, out);
    }
}

// One pair of units a, b on four lanes (hi, lo): lane (e, f) forms s_ef, the four exchange theirs,
// and each has a quarter of the contribution sum_ef g_e m_ef g_f^T: rows hi*HM.., columns lo*HM...
template <typename T, int KP, int GP> struct UnitRaw {
    typedef UnitLayout<T, KP, GP> UL;
    static constexpr int NI = (UL::NP + 3) / 4;
    int4 w[NI];
    __device__ __forceinline__ void load(const char *unit, uint32_t p, int lane)
    {
        const int4 *u = (const int4 *)(unit + (int64_t)p * UL::BYTES);
#pragma unroll
        for (int t = 0; t < NI; t++) w[t] = u[min(4 * t + (lane & 3), UL::NP - 1)];
    }
};
template <typename T, int KP, int GP, bool HI> struct UnitHalf {
    typedef UnitLayout<T, KP, GP> UL;
    union { int4 v[UL::NQ]; double d[KP]; } q;
    union { int4 v[UL::NH]; T d[UL::NH * 16 / sizeof(T)]; int i[UL::NH * 4]; } g;
    __device__ __forceinline__ void take(const UnitRaw<T, KP, GP> &r, bool odd)
    {
        pieces<0, UL::NQ, HI>(r.w, odd, q.v);
        pieces<2 * UL::NQ, UL::NH, HI>(r.w, odd, g.v);
    }
};
template <typename T, int KP, int GP>
__device__ __forceinline__ double unit_dot(const UnitHalf<T, KP, GP, true> &a, const UnitHalf<T, KP, GP, false> &b)
{
    const int sg = a.g.i[UnitLayout<T, KP, GP>::SG / 4];
    double s = 0.0;
    if (__any(sg != 0)) {
#pragma unroll
        for (int k = 0; k < KP; k++) s += (sg >> k) & 1 ? -a.q.d[k] * b.q.d[k] : a.q.d[k] * b.q.d[k];
    } else {
#pragma unroll
        for (int k = 0; k < KP; k++) s = s + a.q.d[k] * b.q.d[k];
    }
    return s;
}
template <typename T, int KP, int GP>
__device__ __forceinline__ void unit_add(const UnitHalf<T, KP, GP, true> &a, const UnitHalf<T, KP, GP, false> &b, double m00,
                                         double m01, double m10, double m11, double (&acc)[GP / 2][GP / 2])
{
    constexpr int HM = GP / 2;
    double b0[HM], b1[HM];
#pragma unroll
    for (int y = 0; y < HM; y++) { b0[y] = (double)b.g.d[y]; b1[y] = (double)b.g.d[HM + y]; }
#pragma unroll
    for (int x = 0; x < HM; x++) {
        const double g0 = (double)a.g.d[x], g1 = (double)a.g.d[HM + x];
        const double t0 = g0 * m00 + g1 * m10, t1 = g0 * m01 + g1 * m11;
#pragma unroll
        for (int y = 0; y < HM; y++) acc[x][y] = acc[x][y] + t0 * b0[y] + t1 * b1[y];
    }
}

// Off-diagonal blocks: SL slots of four lanes per block (16 / SL blocks per wavefront), a slot takes
// every SL-th pair of units of the block; the slots' sums are added in a fixed order at the end.
// Blocks are taken in `perm`'s order: by list length within a window of neighbouring blocks, so the
// blocks of a wavefront have lists of like length.  Units are loaded two pairs ahead.
template <typename T, int KP, int GP, int SL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void k_rows_gather(int64_t nblock /* of this class */, const uint32_t *perm, const int64_t *boff, const int32_t *brg, const int32_t *bcol,
                   const int32_t *gfirst, const uint32_t *ptr, const uint2 *src, const char *unit, double *mat)
{
    // boff null: packed triangle
    constexpr int HM = GP / 2;
    const int lane = threadIdx.x & 63;
    const int64_t p = (xcd_run(blockIdx.x, gridDim.x, 64) * 256 + threadIdx.x) / (4 * SL);
    const int slot = (lane >> 2) & (SL - 1), hi = (lane >> 1) & 1, lo = lane & 1;
    uint32_t i0 = 0, i1 = 0, k = 0;
    int ga = 0, gb = 0;
    if (p < nblock) {
        k = perm[p];
        ga = brg[k];
        gb = bcol[k];
        i0 = ptr[k];
        i1 = ptr[k + 1];
    }
    double acc[HM][HM];
#pragma unroll
    for (int x = 0; x < HM; x++)
#pragma unroll
        for (int y = 0; y < HM; y++) acc[x][y] = 0.0;
    // a0, b0: the current pair; a1, b1: the next; n2: the places of the one after
    UnitRaw<T, KP, GP> a0, b0, a1, b1;
    uint32_t i = i0 + slot;
    uint2 n2 = make_uint2(0, 0);
    const uint32_t last = i1 > 0 ? i1 - 1 : 0;
    if (i1 > i0) {
        const uint2 x = src[min(i, last)], y = src[min(i + SL, last)];
        n2 = src[min(i + 2 * SL, last)];
        a0.load(unit, x.x, lane);
        b0.load(unit, x.y, lane);
        a1.load(unit, y.x, lane);
        b1.load(unit, y.y, lane);
    }
    while (i < i1) {
        UnitHalf<T, KP, GP, true> A;
        UnitHalf<T, KP, GP, false> B;
        A.take(a0, hi);
        B.take(b0, lo);
        a0 = a1;
        b0 = b1;
        a1.load(unit, n2.x, lane);
        b1.load(unit, n2.y, lane);
        n2 = src[min(i + 3 * SL, last)];
        const double s = unit_dot<T, KP, GP>(A, B);
        unit_add<T, KP, GP>(A, B, quad<0x00>(s), quad<0x55>(s), quad<0xaa>(s), quad<0xff>(s), acc);
        i += SL;
    }
    const int nr = gfirst[ga + 1] - gfirst[ga], nc = gfirst[gb + 1] - gfirst[gb];
    const int64_t va = gfirst[ga], vb = gfirst[gb];
    const int64_t m0 = p < nblock && boff ? boff[k] : 0;
#pragma unroll
    for (int x = 0; x < HM; x++)
#pragma unroll
        for (int y = 0; y < HM; y++) {
            double v = acc[x][y];
            if (SL > 1) {
                v += row_ror<4>(v);
                v += row_ror<8>(v);
            }
            if (SL > 4) {
                v += __shfl_xor(v, 16, WV);
                v += __shfl_xor(v, 32, WV);
            }
            const int rr = hi * HM + x, cc = lo * HM + y;
            if (i1 > i0 && slot == ((x * HM + y) & (SL - 1)) && rr < nr && cc < nc) {
                const int64_t i = va + rr;
                mat[boff ? m0 + rr * nc + cc : (i * i - i) / 2 + vb - 1 + cc] -= v;
            }
        }
}

// Diagonal blocks, vector and counters: one workgroup per group, sixteen slots of four lanes in
// each of its wavefronts.  A unit with itself: m_ef = w_e (e = f) - s_ef, and its equations' parts
// of the vector and the counters; two units of one group: -s_ef, both orders.
template <typename T, int KP, int GP>
__global__ __launch_bounds__(256) void k_rows_gather_diag(int32_t ngroup, const int64_t *brow, const int64_t *boff,
                                                          const int32_t *gfirst, const uint32_t *ptr, const uint2 *src,
                                                          const char *unit, const double *side, double *mat, double *vec,
                                                          unsigned long long *cnt)
{
    constexpr int HM = GP / 2;
    __shared__ double s_m[4][GP * GP], s_v[4][GP];
    __shared__ int s_c[4][GP];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int g = blockIdx.x;
    const int64_t k = brow[g + 1] - 1;
    const uint32_t i0 = ptr[k], i1 = ptr[k + 1];
    if (i1 <= i0) return;
    const int slot = lane >> 2, hi = (lane >> 1) & 1, lo = lane & 1;
    double acc[HM][HM], v[HM];
    int c[HM];
#pragma unroll
    for (int x = 0; x < HM; x++) {
        v[x] = 0.0;
        c[x] = 0;
#pragma unroll
        for (int y = 0; y < HM; y++) acc[x][y] = 0.0;
    }
    UnitRaw<T, KP, GP> a, b;
    UnitHalf<T, KP, GP, true> A;
    UnitHalf<T, KP, GP, false> B;
    for (uint32_t i = i0 + wv * 16 + slot; i < i1; i += 64) {
        const uint2 p = src[i];
        a.load(unit, p.x, lane);
        if (p.x == p.y) b = a;
        else b.load(unit, p.y, lane);
        A.take(a, hi);
        B.take(b, lo);
        const double s = -unit_dot<T, KP, GP>(A, B);
        double m00 = quad<0x00>(s), m01 = quad<0x55>(s), m10 = quad<0xaa>(s), m11 = quad<0xff>(s);
        if (p.x == p.y) {
            const double2 w = ((const double2 *)side)[2 * (int64_t)p.x], wr = ((const double2 *)side)[2 * (int64_t)p.x + 1];
            m00 += w.x;
            m11 += w.y;
            unit_add<T, KP, GP>(A, B, m00, m01, m10, m11, acc);
#pragma unroll
            for (int x = 0; x < HM; x++) {
                v[x] = v[x] + wr.x * (double)A.g.d[x] + wr.y * (double)A.g.d[HM + x];
                c[x] += (A.g.d[x] != (T)0) + (A.g.d[HM + x] != (T)0);
            }
        } else {
            unit_add<T, KP, GP>(A, B, m00, m01, m10, m11, acc);
            A.take(b, hi);
            B.take(a, lo);
            unit_add<T, KP, GP>(A, B, m00, m10, m01, m11, acc);
        }
    }
#pragma unroll
    for (int x = 0; x < HM; x++) {
#pragma unroll
        for (int y = 0; y < HM; y++) {
            double t = acc[x][y];
            t += row_ror<4>(t);
            t += row_ror<8>(t);
            t += __shfl_xor(t, 16, WV);
            t += __shfl_xor(t, 32, WV);
            if (slot == 0) s_m[wv][(hi * HM + x) * GP + lo * HM + y] = t;
        }
        double t = v[x];
        int n = c[x];
        for (int o = 4; o < WV; o <<= 1) { t += __shfl_xor(t, o, WV); n += __shfl_xor(n, o, WV); }
        if (slot == 0 && lo == 0) { s_v[wv][hi * HM + x] = t; s_c[wv][hi * HM + x] = n; }
    }
    __syncthreads();
    const int na = gfirst[g + 1] - gfirst[g];
    const int t = threadIdx.x;
    if (t < na * na) {
        const int r = t / na, q = t - r * na;
        const int e = r * GP + q;
        const int64_t v = gfirst[g], i = v + r;
        if (q <= r) mat[boff ? boff[k] + t : (i * i - i) / 2 + v - 1 + q] += (s_m[0][e] + s_m[1][e]) + (s_m[2][e] + s_m[3][e]);
    } else if (t >= 128 && t < 128 + na) {
        const int e = t - 128;
        vec[gfirst[g] - 1 + e] += (s_v[0][e] + s_v[1][e]) + (s_v[2][e] + s_v[3][e]);
        cnt[gfirst[g] - 1 + e] += (unsigned long long)((int64_t)s_c[0][e] + s_c[1][e] + s_c[2][e] + s_c[3][e]);
    }
}

// ---------------------------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------------------------
static unsigned rows_grid(int64_t n, int per, int64_t cap = 1 << 20)
{
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + per - 1) / per, cap));
}

void rows_classify(const StructIn &in, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix,
                   const int32_t *band, const RowGroups &Q, RowStruct &S, std::vector<uint8_t> &cls, hipStream_t s)
{
    const int64_t nrec = in.nrec;
    DBuf<uint8_t> d;
    DBuf<int32_t> mx;
    d.alloc(std::max<int64_t>(nrec, 1));
    S.n.alloc(std::max<int64_t>(4 * nrec, 1));
    mx.alloc(3);
    mx.zero(s);
    cls.assign(nrec, 0);
    int32_t h[3] = {0, 0, 0};
    if (nrec > 0) {
        hipLaunchKernelGGL(k_rows_class, dim3(rows_grid(nrec, RWAVES, 8192)), dim3(WV * RWAVES), 0, s, nrec, in.rec_eq,
                           in.eq_sl, in.eq_n, widx.p, rec_gl.p, gl_tix.p, band, Q, d.p, S.n.p, mx.p);
        HIPCHK(hipGetLastError());
        d.download(cls.data(), nrec, s);
        mx.download(h, 3, s);
    }
    HIPCHK(hipStreamSynchronize(s));
    S.max_eq = h[0];
    S.kp = h[1] <= 2 ? 2 : h[1] <= 4 ? 4 : 6;
    S.gp = h[2] <= 2 ? 2 : h[2] <= 6 ? 6 : 8;
}

#define ROWS_KG(KP_, GP_, F) if (S.kp == KP_ && S.gp == GP_) { F(KP_, GP_); return; }
#define ROWS_ALL(F) \
    ROWS_KG(2, 2, F) ROWS_KG(2, 6, F) ROWS_KG(2, 8, F) ROWS_KG(4, 2, F) ROWS_KG(4, 6, F) ROWS_KG(4, 8, F) \
    ROWS_KG(6, 2, F) ROWS_KG(6, 6, F) ROWS_KG(6, 8, F)

template <typename T>
static void rows_fill_t(const StructIn &in, const T *val, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl,
                        const DBuf<int32_t> &gl_tix, const RowGroups &Q, RowStruct &S, const int64_t *c, hipStream_t s)
{
#define ROWS_F(KP_, GP_)                                                                                                   \
    S.rows.alloc((size_t)std::max<int64_t>(1, S.nrow) * RowLayout<T, KP_, GP_>::RS * sizeof(T));                          \
    hipLaunchKernelGGL((k_rows_fill<T, KP_, GP_>), dim3(rows_grid(S.nq, RWAVES, 8192)), dim3(WV * RWAVES), 0, s, S.nq,     \
                       S.order.p, c, val, in.rec_eq, in.eq_sl, in.eq_n, widx.p, rec_gl.p, gl_tix.p, Q, S.hdr.p,            \
                       (T *)S.rows.p, S.eq_t0.p, S.eq_pos.p, S.seq.p, S.seg.p)
    ROWS_ALL(ROWS_F)
#undef ROWS_F
}

// rows of the records order[0 .. nq) (processing order); the counts' running sums stay in S.c
void rows_build(const StructIn &in, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix,
                const RowGroups &Q, const std::vector<int64_t> &order, RowStruct &S, hipStream_t s)
{
    S.nq = (int64_t)order.size();
    if (S.nq == 0) return;
    S.order.upload(order, s);
    DBuf<int64_t> raw;
    DBuf<uint8_t> tmp;
    const int64_t n1 = S.nq + 1;
    raw.alloc(4 * n1);
    S.c.alloc(4 * n1);
    hipLaunchKernelGGL(k_rows_counts, dim3(rows_grid(n1, 256)), dim3(256), 0, s, S.nq, in.nrec, S.order.p, S.n.p, raw.p);
    size_t bytes = 0;
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, raw.p, S.c.p, (int)n1, s));
    tmp.alloc(std::max<size_t>(bytes, 1));
    int64_t tot[4];
    for (int k = 0; k < 4; k++) {
        HIPCHK(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, raw.p + k * n1, S.c.p + k * n1, (int)n1, s));
        HIPCHK(hipMemcpyAsync(&tot[k], S.c.p + k * n1 + S.nq, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    }
    HIPCHK(hipStreamSynchronize(s));
    S.n.release();
    S.nrow = tot[0];
    S.nseg = tot[1];
    S.nunit = tot[2];
    S.npair = tot[3];
    S.hdr.alloc(S.nq);
    S.eq_t0.alloc(std::max<int64_t>(S.nrow, 1));
    S.eq_pos.alloc(std::max<int64_t>(S.nrow, 1));
    S.seq.alloc(std::max<int64_t>(S.nrow, 1));
    S.seg.alloc(std::max<int64_t>(S.nseg, 1));
    if (in.vd) rows_fill_t<double>(in, in.vd, widx, rec_gl, gl_tix, Q, S, S.c.p, s);
    else rows_fill_t<float>(in, in.vf, widx, rec_gl, gl_tix, Q, S, S.c.p, s);
    HIPCHK(hipGetLastError());
    S.dbl = in.vd != nullptr;
    HIPCHK(hipStreamSynchronize(s));
}

template <typename T> static int unit_bytes_t(const RowStruct &S)
{
#define ROWS_U(KP_, GP_) if (S.kp == KP_ && S.gp == GP_) return UnitLayout<T, KP_, GP_>::BYTES;
    ROWS_U(2, 2) ROWS_U(2, 6) ROWS_U(2, 8) ROWS_U(4, 2) ROWS_U(4, 6) ROWS_U(4, 8) ROWS_U(6, 2) ROWS_U(6, 6) ROWS_U(6, 8)
#undef ROWS_U
    return 0;
}

// batches of the matrix build and their incidence lists: units, their side array and the sort
// buffers of the pairs (24 bytes each) of a batch within `budget` doubles, at most 2^30 pairs.
// upd (when not empty): the size of each record's update, held against the budget instead (a
// budget set by MPGPU_UPDATE_BUFFER_GB counts updates, as it does for the other records)
void rows_incidence(RowStruct &S, const int32_t *group_of, const PairMap &pm, int64_t nblock, const int32_t *brg,
                    const int32_t *bcol, int64_t budget, const std::vector<int64_t> &upd, hipStream_t s)
{
    S.batches.clear();
    if (S.nq == 0) return;
    const int ubytes = S.dbl ? unit_bytes_t<double>(S) : unit_bytes_t<float>(S);
    const int64_t n1 = S.nq + 1, maxpair = (int64_t)1 << 30, ud = ubytes / 8 + 4;
    if (upd.empty() && ud * S.nunit + 3 * S.npair <= budget && S.npair <= maxpair) {
        S.batches.push_back({0, S.nq, 0, S.nunit, 0, S.npair, {0, 0, 0}});
    } else {
        std::vector<int64_t> c(2 * n1);
        HIPCHK(hipMemcpyAsync(c.data(), S.c.p + 2 * n1, sizeof(int64_t) * 2 * n1, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        const int64_t *cu = c.data(), *cp = cu + n1;
        int64_t q0 = 0, inc = 0, size = 0;
        for (int64_t q = 0; q < S.nq; q++) {
            const int64_t d = upd.empty() ? ud * (cu[q + 1] - cu[q]) + 3 * (cp[q + 1] - cp[q]) : upd[q];
            if (q > q0 && (size + d > budget || cp[q + 1] - cp[q0] > maxpair)) {
                S.batches.push_back({q0, q, cu[q0], cu[q] - cu[q0], inc, cp[q] - cp[q0], {0, 0, 0}});
                inc += cp[q] - cp[q0];
                q0 = q;
                size = 0;
            }
            size += d;
        }
        S.batches.push_back({q0, S.nq, cu[q0], S.nunit - cu[q0], inc, S.npair - cp[q0], {0, 0, 0}});
    }
    int64_t mu = 1, mp = 1;
    for (const auto &B : S.batches) {
        mu = std::max(mu, B.nunit);
        mp = std::max(mp, B.npair);
    }
    S.ptr.alloc((size_t)S.batches.size() * (nblock + 1));
    S.src.alloc((size_t)std::max<int64_t>(S.npair, 1));
    DBuf<uint32_t> k0, k1;
    DBuf<uint2> v0;
    DBuf<uint8_t> tmp;
    k0.alloc(mp);
    k1.alloc(mp);
    v0.alloc(mp);
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) <= nblock) bits++;
    size_t bytes = 0;
    HIPCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k0.p, k1.p, v0.p, S.src.p, (int)mp, 0, bits, s));
    tmp.alloc(std::max<size_t>(bytes, 1));
    for (size_t b = 0; b < S.batches.size(); b++) {
        const auto &B = S.batches[b];
        hipLaunchKernelGGL(k_rows_incidence, dim3(rows_grid(B.q1 - B.q0, RWAVES, 8192)), dim3(WV * RWAVES), 0, s, B.q0, B.q1,
                           S.hdr.p, S.seg.p, group_of, pm.bits.p, pm.wrank.p, S.c.p + 3 * n1, B.unit0, k0.p, v0.p);
        if (B.npair > 0)
            HIPCHK(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, k0.p, k1.p, v0.p, S.src.p + B.inc0, (int)B.npair, 0, bits,
                                                      s));
        hipLaunchKernelGGL(k_rows_ptr, dim3(rows_grid(nblock + 1, 256)), dim3(256), 0, s, B.npair, k1.p, nblock,
                           S.ptr.p + b * (nblock + 1));
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(s));
    // order of the blocks in the gather, per batch
    S.perm.alloc(S.batches.size() * (size_t)nblock);
    {
        DBuf<uint64_t> q0, q1;
        DBuf<uint32_t> p0;
        DBuf<unsigned long long> nc;
        DBuf<uint8_t> t2;
        q0.alloc(nblock);
        q1.alloc(nblock);
        p0.alloc(nblock);
        nc.alloc(3 * S.batches.size());
        nc.zero(s);
        HIPCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, q0.p, q1.p, p0.p, S.perm.p, (int)nblock, 0, 38, s));
        t2.alloc(std::max<size_t>(bytes, 1));
        for (size_t b = 0; b < S.batches.size(); b++) {
            hipLaunchKernelGGL(k_rows_len, dim3(rows_grid(nblock, 256, 2048)), dim3(256), 0, s, nblock, S.ptr.p + b * (nblock + 1), brg,
                               bcol, q0.p, p0.p, nc.p + 3 * b);
            HIPCHK(hipcub::DeviceRadixSort::SortPairs(t2.p, bytes, q0.p, q1.p, p0.p, S.perm.p + b * nblock, (int)nblock, 0, 38, s));
        }
        std::vector<unsigned long long> h(3 * S.batches.size());
        nc.download(h.data(), h.size(), s);
        HIPCHK(hipStreamSynchronize(s));
        for (size_t b = 0; b < S.batches.size(); b++)
            for (int x = 0; x < 3; x++) S.batches[b].ncls[x] = (int64_t)h[3 * b + x];
    }
    S.unit_bytes = (size_t)mu * ubytes;
    S.side_len = (size_t)mu * 4;
    S.alloc_units();
    S.c.release();
}

template <typename T, int KP, int GP, bool BUILD>
static hipError_t rows_launch(const RowDev &R, const DevModel &M, const PassOpts &o, const RecOut &out, int64_t q0, int64_t q1,
                              int max_eq, hipStream_t s)
{
    const int mq = max_eq <= WV ? WV : MAXEQ;
    const int lds = rows_lds<T, KP, GP>(mq, BUILD) * RWAVES;
    hipError_t e;
    if (lds > 65536) {
        e = hipFuncSetAttribute((const void *)k_rows_pass<T, KP, GP, BUILD>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    // as many workgroups as fit on the device at once; each loops over the records
    int per_cu = 0, dev = 0, ncu = 0;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_rows_pass<T, KP, GP, BUILD>, WV * RWAVES, lds)) != hipSuccess)
        return e;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    const int grid = (int)std::min<int64_t>((q1 - q0 + RWAVES - 1) / RWAVES, (int64_t)std::max(1, per_cu) * std::max(1, ncu));
    hipLaunchKernelGGL((k_rows_pass<T, KP, GP, BUILD>), dim3(std::max(1, grid)), dim3(WV * RWAVES), lds, s, R, M, o, out, q0, q1, mq);
    return hipGetLastError();
}

hipError_t launch_rows(const RowStruct &S, const RowDev &R, const DevModel &M, const PassOpts &o, const RecOut &out, bool build,
                       int64_t q0, int64_t q1, hipStream_t s)
{
    if (q1 <= q0) return hipSuccess;
#define ROWS_L(KP_, GP_)                                                                                                  \
    if (S.kp == KP_ && S.gp == GP_) {                                                                                     \
        if (S.dbl)                                                                                                        \
            return build ? rows_launch<double, KP_, GP_, true>(R, M, o, out, q0, q1, S.max_eq, s)                         \
                         : rows_launch<double, KP_, GP_, false>(R, M, o, out, q0, q1, S.max_eq, s);                       \
        return build ? rows_launch<float, KP_, GP_, true>(R, M, o, out, q0, q1, S.max_eq, s)                              \
                     : rows_launch<float, KP_, GP_, false>(R, M, o, out, q0, q1, S.max_eq, s);                            \
    }
    ROWS_L(2, 2) ROWS_L(2, 6) ROWS_L(2, 8) ROWS_L(4, 2) ROWS_L(4, 6) ROWS_L(4, 8) ROWS_L(6, 2) ROWS_L(6, 6) ROWS_L(6, 8)
#undef ROWS_L
    return hipErrorInvalidValue;
}

hipError_t launch_rows_gather(const RowStruct &S, size_t batch, int32_t ngroup, int64_t nblock,
                              const int64_t *brow, const int64_t *boff, const int32_t *brg, const int32_t *bcol,
                              const int32_t *gfirst, double *mat, double *vec, unsigned long long *cnt, hipStream_t s)
{
    if (nblock <= 0) return hipSuccess;
    const auto &B = S.batches[batch];
    const uint32_t *ptr = S.ptr.p + batch * (nblock + 1);
    const uint2 *src = S.src.p + B.inc0;
    const uint32_t *perm = S.perm.p + batch * nblock;
#define ROWS_GS(T_, KP_, GP_, SL_, N_)                                                                                     \
    if ((N_) > 0) {                                                                                                       \
        hipLaunchKernelGGL((k_rows_gather<T_, KP_, GP_, SL_>), dim3((unsigned)(((N_) * 4 * SL_ + 255) / 256)), dim3(256), \
                           0, s, N_, perm, boff, brg, bcol, gfirst, ptr, src, (const char *)S.unit.p, mat);               \
        perm += (N_);                                                                                                     \
    }
#define ROWS_G(T_, KP_, GP_)                                                                                               \
    if (S.kp == KP_ && S.gp == GP_) {                                                                                     \
        ROWS_GS(T_, KP_, GP_, 16, B.ncls[0]) ROWS_GS(T_, KP_, GP_, 4, B.ncls[1]) ROWS_GS(T_, KP_, GP_, 1, B.ncls[2])      \
        hipLaunchKernelGGL((k_rows_gather_diag<T_, KP_, GP_>), dim3(ngroup), dim3(256), 0, s, ngroup, brow, boff, gfirst, \
                           ptr, src, (const char *)S.unit.p, S.side.p, mat, vec, cnt);                                    \
    }
#define ROWS_GT(T_) \
    ROWS_G(T_, 2, 2) ROWS_G(T_, 2, 6) ROWS_G(T_, 2, 8) ROWS_G(T_, 4, 2) ROWS_G(T_, 4, 6) ROWS_G(T_, 4, 8) \
    ROWS_G(T_, 6, 2) ROWS_G(T_, 6, 6) ROWS_G(T_, 6, 8)
    if (S.dbl) { ROWS_GT(double) } else { ROWS_GT(float) }
#undef ROWS_G
#undef ROWS_GS
#undef ROWS_GT
    return hipGetLastError();
}

} // namespace mpgpu
