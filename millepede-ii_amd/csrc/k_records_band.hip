// Record-loop kernel for local fits with bordered-band structure: one workgroup of 256
// threads per record.
//
// Restates loopbf (src/pede.f90:3387-4442) for the records whose local normal matrix pede
// solves with sqmibb / sqmibb2 (src/mpnum.f90:3118-3628): a band of half-width mbnd plus mbdr
// border rows at the start (side 1) or at the end (side 2), as chosen per record by the cost
// model of src/pede.f90:3838-3874 (evaluated on the host when the structure is built).
//
//  * the local matrix is accumulated directly into band and border storage (equations in
//    order, the same per-element arithmetic as the full path);
//  * root-free band Cholesky (dbcdec), band solves for the border columns and the right-hand
//    side (dbcslv), border Schur complement inverted with sqminv, back-substitution - the
//    operation order of sqmibb, so rank and condition decisions are pede's;
//  * the complete inverse (inv = 2) is formed column by column from the right with the dbcinv
//    recursion (the entries of a column need only the mbnd columns to its right, held in an
//    LDS ring), plus the border corrections, into LDS where it fits beside the rest, else into a
//    per-workgroup global scratch area;
//  * G Gamma^-1 G^T (dbavats order, src/mpnum.f90:1470-1528) uses support classes: runs of
//    record globals whose rows of G have the same local-parameter support share the same
//    block of Gamma^-1, so each matrix element costs |S| FMAs and one FP64 atomic.
//
// Chains of dependent steps bound it (equation after equation, column after column), so one
// wavefront walks the short ones with LDS order instead of workgroup barriers and with the words of
// the next four equations in flight, and as many records as possible are in flight beside each
// other: 128 registers for four workgroups a CU, though some values spill (three without spills: 8.4
// against 5.4 ms), and a grid of what is resident.  20,000 broken-lines tracks of up to 44 local
// parameters: 12.2 -> 5.3 ms.
#include "mpgpu_device.h"
#include <float.h>

namespace mpgpu {

#define BNT 256
#define BWAVES (BNT / 64)
#define QCH 16         // support entries of one class handled per register chunk

__device__ __forceinline__ int64_t bpk64(int64_t i, int64_t j) { return (i * i - i) / 2 + j - 1; }
// packed index of (i, j) in either order, 1-based
__device__ __forceinline__ int64_t bsym(int i, int j) { return i >= j ? bpk64(i, j) : bpk64(j, i); }

template <typename T> __device__ __forceinline__ double bval(const DevRecords &R, int64_t w);
template <> __device__ __forceinline__ double bval<float>(const DevRecords &R, int64_t w) { return (double)R.vf[w]; }
template <> __device__ __forceinline__ double bval<double>(const DevRecords &R, int64_t w) { return R.vd[w]; }

__device__ __forceinline__ void band_mat_add(const DevModel &M, int va, int vb, double v, const int32_t *seg_of,
                                             const int2 *seg_fn, const int32_t *pblk, int pos_a, int pos_b)
{
    if (!M.sparse) {
        atomicAdd(&M.mat[bpk64(va, vb)], v);
    } else {
        int sa = seg_of[pos_a], sb = seg_of[pos_b];
        int blk = pblk[(sa * sa + sa) / 2 + sb];
        if (blk < 0) return;
        atomicAdd(&M.mat[M.boff[blk] + (int64_t)(va - seg_fn[sa].x) * seg_fn[sb].y + (vb - seg_fn[sb].x)], v);
    }
}

// block-wide sum (all threads return the total)
__device__ double block_sum(double v, double *red)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < BWAVES; k++) s += red[k];
    __syncthreads();
    return s;
}

// symmetric Gauss-Jordan with diagonal pivoting (sqminv, src/mpnum.f90:97-213), one thread,
// on a small packed matrix (the border Schur complement); 1-based v, b
__device__ void sqminv_small(double *v, double *b, int n, int *nrank, double *diag, int *next)
{
    const double eps = 16.0 * DBL_EPSILON;
    int next0 = 1, l = 1;
    for (int i = 1; i <= n; i++) {
        next[i] = i + 1;
        diag[i] = fabs(v[(i * i + i) / 2]);
    }
    next[n] = -1;
    *nrank = 0;
    for (int i = 1; i <= n; i++) {
        int k = 0;
        double vkk = 0.0;
        int j = next0, last = 0;
        while (j > 0) {
            int jj = (j * j + j) / 2;
            double m = fabs(vkk) > eps * diag[j] ? fabs(vkk) : eps * diag[j];
            if (fabs(v[jj]) > m) { vkk = v[jj]; k = j; l = last; }
            last = j;
            j = next[last];
        }
        if (k != 0) {
            int kk = (k * k + k) / 2;
            if (l == 0) next0 = next[k]; else next[l] = next[k];
            next[k] = 0;
            (*nrank)++;
            vkk = 1.0 / vkk;
            v[kk] = -vkk;
            b[k] = b[k] * vkk;
            int jk = kk - k, jl = 0;
            for (int jx = 1; jx <= n; jx++) {
                if (jx == k) { jk = kk; jl = jl + jx; }
                else {
                    if (jx < k) jk = jk + 1; else jk = jk + jx - 1;
                    double vjk = v[jk];
                    v[jk] = vkk * vjk;
                    b[jx] = b[jx] - b[k] * vjk;
                    int lk = kk - k;
                    for (int lx = 1; lx <= jx; lx++) {
                        jl = jl + 1;
                        if (lx == k) lk = kk;
                        else {
                            if (lx < k) lk = lk + 1; else lk = lk + lx - 1;
                            v[jl] = v[jl] - v[lk] * vjk;
                        }
                    }
                }
            }
        } else {
            for (int kx = 1; kx <= n; kx++) {
                if (next[kx] != 0) {
                    b[kx] = 0.0;
                    for (int jx = 1; jx <= kx; jx++)
                        if (next[jx] != 0) v[(kx * kx - kx) / 2 + jx] = 0.0;
                }
            }
            break;
        }
    }
    for (int i = 1; i <= (n * n + n) / 2; i++) v[i] = -v[i];
}

// Equations in order, 64 at a time, by one wavefront: lane q gets word q of the equation (its local
// or total position and its value), the words of the next equations are in flight, and
// f(i, words) does equation i.  Every equation has at most 64 words.
template <typename T> struct EqWords { int nl, ng, wx; T v; };
template <typename T> __device__ __forceinline__ T raw_val(const DevRecords &R, int64_t w);
template <> __device__ __forceinline__ float raw_val<float>(const DevRecords &R, int64_t w) { return R.vf[w]; }
template <> __device__ __forceinline__ double raw_val<double>(const DevRecords &R, int64_t w) { return R.vd[w]; }
__device__ __forceinline__ double lane_val(float v, int l) { return (double)__shfl(v, l, 64); }
__device__ __forceinline__ double lane_val(double v, int l) { return __shfl(v, l, 64); }
template <typename T, class F>
__device__ __forceinline__ void each_equation(const DevRecords &R, int64_t e0, int neq, int lane, F f)
{
    constexpr int D = 4;                                   // equations in flight
    for (int base = 0; base < neq; base += 64) {
        const int ne = min(64, neq - base);
        const int64_t slv = R.eq_sl[e0 + base + min(lane, ne - 1)];
        const uint32_t env = R.eq_n[e0 + base + min(lane, ne - 1)];
        EqWords<T> W[D];
        auto ld = [&](int i, EqWords<T> &E) {
            const int q = min(i, ne - 1);
            const int64_t sl = ((int64_t)__builtin_amdgcn_readlane((int)(slv >> 32), q) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)slv, q);
            const uint32_t en = (uint32_t)__builtin_amdgcn_readlane((int)env, q);
            E.nl = en & 0xffff;
            E.ng = en >> 16;
            const int64_t w = sl + min(lane, E.nl + E.ng + 1);
            E.wx = R.widx[w];
            E.v = raw_val<T>(R, w);
        };
#pragma unroll
        for (int u = 0; u < D; u++) ld(u, W[u]);
        for (int i = 0; i < ne; i += D) {
#pragma unroll
            for (int u = 0; u < D; u++) {
                if (i + u < ne) f(base + i + u, W[u]);
                ld(i + u + D, W[u]);
            }
        }
    }
}

// band solve with the root-free factor (dbcslv, src/Dbandmatrix.f90:521-560), one thread;
// w column-major w(mp1, n) 1-based through W(r, c) = w[(c - 1) * mp1 + r]; x 1-based, in place
__device__ void dbcslv_any(const double *w, int mp1, int n, double *x)
{
    for (int i = 1; i <= n; i++) {
        const double xi = x[i];
        const int jm = min(mp1 - 1, n - i);
        for (int j = 1; j <= jm; j++) x[j + i] = x[j + i] - w[(i - 1) * mp1 + j + 1] * xi;
    }
    for (int i = n; i >= 1; i--) {
        double rxw = x[i] * w[(i - 1) * mp1 + 1];
        const int jm = min(mp1 - 1, n - i);
        for (int j = 1; j <= jm; j++) rxw = rxw - w[(i - 1) * mp1 + j + 1] * x[j + i];
        x[i] = rxw;
    }
}

// the same for a half-width of at most MB: the last MB solutions in registers, so that the chain
// from one row to the next has no LDS access (the loads run ahead of it); the terms of a row come
// in the same order
template <int MB>
__device__ void dbcslv_win(const double *w, int mp1, int n, double *x)
{
    double xw[MB];
#pragma unroll
    for (int j = 0; j < MB; j++) xw[j] = 0.0;
    for (int i = 1; i <= n; i++) {
        double v = x[i];
#pragma unroll
        for (int j = MB; j >= 1; j--) {                    // sources i - MB .. i - 1
            const bool ok = j < mp1 && j < i;
            const double c = w[ok ? (i - j - 1) * mp1 + j + 1 : 1];
            v = v - (ok ? c : 0.0) * xw[j - 1];
        }
#pragma unroll
        for (int j = MB - 1; j >= 1; j--) xw[j] = xw[j - 1];
        xw[0] = v;
        x[i] = v;
    }
#pragma unroll
    for (int j = 0; j < MB; j++) xw[j] = 0.0;
    for (int i = n; i >= 1; i--) {
        double v = x[i] * w[(i - 1) * mp1 + 1];
#pragma unroll
        for (int j = 1; j <= MB; j++) {
            const bool ok = j < mp1 && i + j <= n;
            const double c = w[ok ? (i - 1) * mp1 + j + 1 : 1];
            v = v - (ok ? c : 0.0) * xw[j - 1];
        }
#pragma unroll
        for (int j = MB - 1; j >= 1; j--) xw[j] = xw[j - 1];
        xw[0] = v;
        x[i] = v;
    }
}
__device__ void dbcslv_thread(const double *w, int mp1, int n, double *x)
{
    if (mp1 <= 7) dbcslv_win<6>(w, mp1, n, x);
    else dbcslv_any(w, mp1, n, x);
}

template <typename T, bool VL>
__global__ __launch_bounds__(BNT, 4) void k_records_band(DevRecords R, DevModel M, PassOpts o, RecOut out, BandPlan P,
                                                      const int64_t *ids, int64_t nb, const int32_t *binfo,
                                                      double *scratch)
{
    extern __shared__ double lds[];
    const int tid = threadIdx.x;
    const double chuber = 1.345, cauchy = 2.3849;
    const int NA = P.nalc_max;

    // ---- carve LDS (1-based arrays get one spare element) ----
    double *gp = lds;                              // [max_gl]
    double *rm = gp + P.max_gl;                    // [max_eq]
    double *re = rm + P.max_eq;
    double *lc = re + P.max_eq;
    double *lw = lc + P.max_eq;
    double *vbnd = lw + P.max_eq;                  // [NA*mp1_max + 1] band, W(r,c) = vbnd[(c-1)*mp1 + r]
    double *vbdr = vbnd + NA * P.mp1_max + 1;      // [nbdr_max*NA + 1]
    double *aux = vbdr + P.nbdr_max * NA + 1;      // [nbdr_max*NA + NA + 1]
    double *bl = aux + (P.nbdr_max + 1) * NA + 1;  // [NA + 1]
    double *bs = bl + NA + 1;                      // [NA + 1]
    double *vbk = bs + NA + 1;                     // [nbdr_max(nbdr_max+1)/2 + 1]
    double *vzru = vbk + (P.nbdr_max * P.nbdr_max + P.nbdr_max) / 2 + 1; // [nbdr_max + 1]
    double *sdiag = vzru + P.nbdr_max + 1;         // [nbdr_max + 1]
    double *ring = sdiag + P.nbdr_max + 1;         // [mp1_max * (NA + 1)]
    double *gval = ring + P.mp1_max * (NA + 1);    // [max_sup]
    double *red = gval + P.max_sup;                // [8]
    unsigned long long *mask = (unsigned long long *)(red + 8); // [max_var * nwm]
    int32_t *gv = (int32_t *)(mask + (size_t)P.max_var * P.nwm);  // [max_gl]
    int32_t *gpos = gv + P.max_gl;                 // [max_gl]
    int32_t *gvl = gpos + P.max_gl;                // [max_var]
    int32_t *segof = gvl + P.max_var;              // [max_var]
    int32_t *clsof = segof + P.max_var;            // [max_var]
    int32_t *gptr = clsof + P.max_var;             // [max_var + 1]
    int32_t *cls0 = gptr + P.max_var + 1;          // [max_var + 1] first global of each class
    int32_t *sptr = cls0 + P.max_var + 1;          // [max_var + 1] support offsets of each class
    int32_t *upre = sptr + P.max_var + 1;          // [max_var + 1] work-unit prefix per class
    int32_t *sidx = upre + P.max_var + 1;          // [max_sup] support (local indices) of each class
    int32_t *pblk = sidx + P.max_sup;              // [max_pair]
    int32_t *snext = pblk + P.max_pair;            // [nbdr_max + 1]
    int32_t *sh = snext + P.nbdr_max + 1;          // [32] scalars

    // packed inverse, 0-based bpk64
    double *vinv;
    if constexpr (VL) vinv = lds + P.vinv_lds;
    else vinv = scratch + (size_t)blockIdx.x * P.vinv_stride;
    const int nwm = P.nwm;
    int2 *segfn = (int2 *)gp;                      // first variable and size of each segment's group (gp is done by then)
    // pair (pj, pk), pj >= pk, of lane tid in the packed triangle
    int pj = 1, pk = 1;
    {
        int rem = tid & 63;
        while (rem >= pj) rem -= pj++;
        pk = rem + 1;
    }

    for (int64_t ri = blockIdx.x; ri < nb; ri += gridDim.x) {
        const int64_t r = ids[ri];
        const int32_t info = binfo[r];
        const int mbnd = (info & 0x3ff) - 1, mbdr = (info >> 10) & 0x3ff, mside = (info >> 20) & 3;
        const int64_t e0 = R.rec_eq[r];
        const int neq = (int)(R.rec_eq[r + 1] - e0);
        const int64_t g0 = R.rec_gl[r];
        const int ngl = (int)(R.rec_gl[r + 1] - g0);
        const double dw1 = R.rec_w ? (double)R.rec_w[r] : 1.0;
        const double dw2 = sqrt(dw1);
        if (neq > P.max_eq || ngl > P.max_gl || mbnd + 1 > P.mp1_max || mbdr > P.nbdr_max) {
            if (tid == 0) { out.status[r] = 9; out.chi2[r] = 0.0; out.ndf[r] = 0; }
            continue;
        }
        // ---- distinct labels (wave 0) ----
        if (tid < 64) {
            int nalg = 0;
            for (int base = 0; base < ngl; base += 64) {
                int k = base + tid;
                int v = 0;
                if (k < ngl) {
                    int t = R.gl_tix[g0 + k];
                    gp[k] = M.par[t];
                    v = M.var[t];
                    gv[k] = v;
                }
                bool isv = (k < ngl) && v > 0;
                unsigned long long m = __ballot(isv);
                int pos = nalg + __popcll(m & ((1ull << tid) - 1ull));
                if (k < ngl) gpos[k] = isv ? pos : -1;
                if (isv && pos < P.max_var) gvl[pos] = v;
                nalg += __popcll(m);
            }
            if (tid == 0) { sh[0] = nalg; sh[1] = 0; sh[7] = 0; }
        }
        __syncthreads();
        const int nalg = sh[0];
        // ---- first loop: residuals after the global parameters, number of locals ----
        for (int i = tid; i < neq; i += BNT) {
            int64_t sl = R.eq_sl[e0 + i];
            uint32_t en = R.eq_n[e0 + i];
            int nl = en & 0xffff, ng = en >> 16;
            int64_t sg = sl + nl + 1;
            double rmeas = bval<T>(R, sl);
            for (int j = 1; j <= ng; j++) rmeas = rmeas - bval<T>(R, sg + j) * gp[R.widx[sg + j]];
            rm[i] = rmeas;
            // 'scaleerrors' (prepareRecords, src/mppar.f90:312-316)
            re[i] = bval<T>(R, sg) * (ng > 0 ? o.esc[0] : o.esc[1]);
            lc[i] = 0.0;
            int mx = 0;
            for (int j = 1; j <= nl; j++) mx = max(mx, R.widx[sl + j]);
            if (mx > 0) atomicMax(&sh[1], mx);
            if (nl > 9 || nl + ng + 2 > 64) atomicOr(&sh[7], 1);
        }
        __syncthreads();
        const int nalc = sh[1];
        const int nmb = nalc - mbdr, mp1 = mbnd + 1;
        // equations of at most 64 words and 9 locals, a band of at most 64 rows and 10 columns: one
        // wavefront does the serial phases without workgroup barriers
        const bool eq1 = sh[7] == 0, one = nmb <= 64 && mbnd <= 10;
        const int tn = one ? 64 : BNT;
        auto tsync = [&]() {
            if (one) wave_order();
            else __syncthreads();
        };
        if (nalg > P.max_var || nalc > NA || nalc <= 0 || nmb <= 0) {
            if (tid == 0) { out.status[r] = 9; out.chi2[r] = 0.0; out.ndf[r] = 0; }
            __syncthreads();
            continue;
        }
        const int nb1 = mside == 1 ? mbdr + 1 : nmb + 1;     // first band (side 1) / border (side 2) index
        const int bo = mside == 1 ? mbdr : 0;                  // band offset in local numbering
        // ---- local fit iterations (3759-4094) ----
        const int nter = (o.nloopn != 1 && o.lhuber != 0) ? o.lhuber : 1;
        int status = 0, nrank = 0, ndf = 0;
        double summ = 0.0;
        float resing = 0.0f;
        for (int iter = 1; iter <= nter; iter++) {
            for (int i = tid; i < neq; i += BNT) {
                double rerr = re[i];
                double wght = 1.0 / (rerr * rerr);
                double resid = rm[i] - lc[i];
                if (o.nloopn != 1 && iter != 1 && o.lhuber != 0) {
                    if (iter <= 3) {
                        if (fabs(resid) > chuber * rerr) wght = wght * chuber * rerr / fabs(resid);
                    } else {
                        double t = resid / rerr / cauchy;
                        wght = wght / (1.0 + t * t);
                    }
                }
                lw[i] = wght;
            }
            for (int t = tid; t < nmb * mp1 + 1; t += BNT) vbnd[t] = 0.0;
            for (int t = tid; t < mbdr * nalc + 1; t += BNT) vbdr[t] = 0.0;
            for (int t = tid; t <= nalc; t += BNT) bl[t] = 0.0;
            if (tid == 0) sh[2] = 0;
            __syncthreads();
            // local normal equations into band / border storage, equations in order
            auto put = [&](int ij, int ik, double val) {
                const int J = max(ij, ik), K = min(ij, ik);
                if (mside == 1) {
                    if (K <= mbdr) vbdr[(K - 1) * nalc + J] += val;          // column K of the border
                    else if (J - K <= mbnd) vbnd[(K - nb1) * mp1 + J - K + 1] += val;
                    else sh[2] = 1;
                } else {
                    if (J > nmb) vbdr[(J - nb1) * nalc + K] += val;           // row J of the border
                    else if (J - K <= mbnd) vbnd[(K - 1) * mp1 + J - K + 1] += val;
                    else sh[2] = 1;
                }
            };
            if (eq1 && tid < 64)
                each_equation<T>(R, e0, neq, tid, [&](int i, const EqWords<T> &E) {
                    const int npair = (E.nl * E.nl + E.nl) / 2;
                    const bool rhs = tid >= 64 - E.nl;     // the last lanes: the right-hand side
                    const int j = rhs ? 64 - tid : pj, k = pk;
                    const int ij = __shfl(E.wx, j, 64), ik = __shfl(E.wx, k, 64);
                    const double vj = lane_val(E.v, j), vk = lane_val(E.v, k);
                    const double wght = lw[i];
                    if (rhs) bl[ij] = bl[ij] + wght * rm[i] * vj;
                    else if (tid < npair) put(ij, ik, wght * vj * vk);
                    wave_order();
                });
            for (int i = 0; i < (eq1 ? 0 : neq); i++) {
                const int64_t sl = R.eq_sl[e0 + i];
                const int nl = R.eq_n[e0 + i] & 0xffff;
                const int npair = (nl * nl + nl) / 2;
                const double wght = lw[i];
                for (int t = tid; t < npair + nl; t += BNT) {
                    if (t >= npair) {
                        int j = t - npair + 1;
                        int ij = R.widx[sl + j];
                        bl[ij] = bl[ij] + wght * rm[i] * bval<T>(R, sl + j);
                        continue;
                    }
                    int j = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5) + 1;
                    while ((j * j - j) / 2 > t) j--;
                    while ((j * j + j) / 2 <= t) j++;
                    int k = t - (j * j - j) / 2 + 1;
                    int ij = R.widx[sl + j], ik = R.widx[sl + k];
                    double val = wght * bval<T>(R, sl + j) * bval<T>(R, sl + k);
                    put(ij, ik, val);
                }
                __syncthreads();
            }
            __syncthreads();
            if (sh[2]) { status = 9; break; }   // element outside the detected structure
            // ---- sqmibb / sqmibb2: root-free band Cholesky (dbcdec) ----
            for (int i = tid; i < nmb; i += BNT) aux[i + 1] = 16.0 * vbnd[i * mp1 + 1];
            __syncthreads();
            if (tid < tn) {
                for (int i = 1; i <= nmb; i++) {
                    const int jm = min(mp1 - 1, nmb - i);
                    double piv = vbnd[(i - 1) * mp1 + 1];
                    piv = (piv + aux[i] != aux[i]) ? 1.0 / piv : 0.0;
                    // W(k, i+j) -= W(k+j, i) * rxw, rxw = W(j+1, i) * W(1, i); pairs (j, k) independent
                    // (pair (pj, pk) of the triangle: j = pk, k + j = pj)
                    int j = pk, kj = pj;
                    if (!one) {
                        kj = 1;
                        int rem = tid;
                        while (rem >= kj) rem -= kj++;
                        j = rem + 1;
                    }
                    double upd = 0.0;
                    int tgt = -1;
                    if (kj <= jm) {
                        const double rxw = vbnd[(i - 1) * mp1 + j + 1] * piv;
                        tgt = (i + j - 1) * mp1 + kj - j + 1;
                        upd = vbnd[tgt] - vbnd[(i - 1) * mp1 + kj + 1] * rxw;
                    }
                    tsync();
                    if (tgt >= 0) vbnd[tgt] = upd;
                    if (tid < jm) vbnd[(i - 1) * mp1 + tid + 2] = vbnd[(i - 1) * mp1 + tid + 2] * piv;
                    if (tid == 0) vbnd[(i - 1) * mp1 + 1] = piv;
                    tsync();
                }
            }
            __syncthreads();
            // rank of the band part and its condition (inverted pivots, as sqmibb)
            if (tid == 0) {
                int ok = 1;
                double emin = 0.0, emax = 0.0;
                for (int i = 1; i <= nmb; i++) {
                    double d = vbnd[(i - 1) * mp1 + 1];
                    if (d <= 0.0) { ok = 0; break; }
                    if (i == 1) { emin = d; emax = d; }
                    else { emin = fmin(emin, d); emax = fmax(emax, d); }
                }
                sh[3] = ok;
                red[4] = emin;
                red[5] = emax;
            }
            __syncthreads();
            const bool bandok = sh[3] != 0;
            const double evdmin = red[4], evdmax = red[5];
            __syncthreads();
            int nrankb = 0;
            if (!bandok) {
                for (int t = tid; t <= nalc; t += BNT) bl[t] = 0.0;
                nrank = 0;
                __syncthreads();
            } else if (mbdr == 0) {
                if (tid == 0) dbcslv_thread(vbnd, mp1, nmb, bl);
                nrank = nmb;
                __syncthreads();
            } else {
                // border columns and the band part of the right-hand side, one thread each
                const int n = nalc;
                if (tid < mbdr) {
                    const int ib = tid + 1;
                    double *ax = (mside == 1) ? &aux[nb1 + (ib - 1) * n - 1] : &aux[(ib - 1) * n];
                    const double *src = (mside == 1) ? &vbdr[nb1 + (ib - 1) * n - 1] : &vbdr[(ib - 1) * n];
                    for (int i = 1; i <= nmb; i++) ax[i] = src[i];
                    dbcslv_thread(vbnd, mp1, nmb, ax);
                } else if (tid == mbdr) {
                    const double *src = (mside == 1) ? &bl[nb1 - 1] : &bl[0];
                    for (int i = 1; i <= nmb; i++) bs[i] = src[i];
                    dbcslv_thread(vbnd, mp1, nmb, bs);
                }
                __syncthreads();
                // VZRU = b_border - AUX^T b_band (original b), VBK = C_bb - C_bn AUX
                const int nq = (mbdr * mbdr + mbdr) / 2;
                if (tid < mbdr) {
                    const int ib = tid + 1;
                    double z;
                    if (mside == 1) {
                        const int ioff = nb1 + (ib - 1) * n;
                        z = bl[ib];
                        for (int i = 0; i <= nmb - 1; i++) z = z - bl[nb1 + i] * aux[ioff + i];
                    } else {
                        const int ioff = (ib - 1) * n;
                        z = bl[nmb + ib];
                        for (int i = 1; i <= nmb; i++) z = z - bl[i] * aux[ioff + i];
                    }
                    vzru[ib] = z;
                } else if (tid >= 64 && tid < 64 + nq) {
                    int q = tid - 64 + 1, ib = 1;
                    while ((ib * ib + ib) / 2 < q) ib++;
                    const int jb = q - (ib * ib - ib) / 2;
                    double s;
                    if (mside == 1) {
                        const int ioff = nb1 + (ib - 1) * n, joff = nb1 + (jb - 1) * n;
                        s = vbdr[(jb - 1) * n + ib];
                        for (int i = 0; i <= nmb - 1; i++) s = s - vbdr[ioff + i] * aux[joff + i];
                    } else {
                        const int ioff = (ib - 1) * n, joff = (jb - 1) * n;
                        s = vbdr[(ib - 1) * n + nmb + jb];
                        for (int i = 1; i <= nmb; i++) s = s - vbdr[ioff + i] * aux[joff + i];
                    }
                    vbk[q] = s;
                }
                __syncthreads();
                if (tid == 0) {
                    int nr = 0;
                    sqminv_small(vbk, vzru, mbdr, &nr, sdiag, snext);
                    if (nr != mbdr) {
                        for (int ib = 1; ib <= mbdr; ib++) vzru[ib] = 0.0;
                        for (int q = 1; q <= nq; q++) vbk[q] = 0.0;
                    }
                    sh[4] = nr;
                }
                __syncthreads();
                nrankb = sh[4];
                nrank = nmb + (nrankb == mbdr ? mbdr : 0);
                // back-substitution of the band part with the border solution
                for (int i = tid + 1; i <= nmb; i += BNT) {
                    double x = bs[i];
                    if (mside == 1) {
                        for (int ib = 1; ib <= mbdr; ib++) x = x - vzru[ib] * aux[nb1 + (ib - 1) * n + i - 1];
                        bl[nb1 + i - 1] = x;
                    } else {
                        for (int ib = 1; ib <= mbdr; ib++) x = x - vzru[ib] * aux[(ib - 1) * n + i];
                        bl[i] = x;
                    }
                }
                if (tid < mbdr) bl[(mside == 1 ? 0 : nmb) + tid + 1] = vzru[tid + 1];
                __syncthreads();
            }
            float cndl10 = 0.0f;
            if (bandok && evdmin > 0.0) cndl10 = log10f((float)(evdmax / evdmin));
            // NaN check and third loop: residuals, chi^2 (3903-4035)
            int nan = 0;
            for (int i = tid + 1; i <= nalc; i += BNT) {
                double b = bl[i];
                if (!(b <= 0.0) && !(b > 0.0)) nan++;
            }
            double s_chi = 0.0, s_wt = 0.0;
            for (int i = tid; i < neq; i += BNT) {
                int64_t sl = R.eq_sl[e0 + i];
                int nl = R.eq_n[e0 + i] & 0xffff;
                double rerr = re[i];
                double wght = 1.0 / (rerr * rerr);
                double rmloc = 0.0;
                for (int j = 1; j <= nl; j++) rmloc = rmloc + bval<T>(R, sl + j) * bl[R.widx[sl + j]];
                lc[i] = rmloc;
                double rmeas = rm[i] - rmloc;
                double dchi2 = wght * rmeas * rmeas;
                double resid = rmeas;
                if (o.nloopn != 1 && iter != 1 && o.lhuber != 0) {
                    if (iter <= 3) {
                        if (fabs(resid) > chuber * rerr) {
                            wght = wght * chuber * rerr / fabs(resid);
                            dchi2 = 2.0 * chuber * (fabs(resid) / rerr - 0.5 * chuber);
                        }
                    } else {
                        double t = resid / rerr / cauchy;
                        wght = wght / (1.0 + t * t);
                        dchi2 = log(1.0 + t * t) * cauchy * cauchy;
                    }
                }
                double down = 1.0 / sqrt(wght);
                s_wt += rerr / down;
                s_chi += dchi2;
                if (iter == nter) rm[i] = rmeas;
            }
            nan = (int)block_sum((double)nan, red);
            summ = block_sum(s_chi, red);
            double suwt = block_sum(s_wt, red);
            ndf = neq - nrank;
            resing = ((float)neq - (float)suwt) / (float)neq;
            if (nan > 0) { status = 1; break; }
            if (nrank != nalc) { status = 2; break; }
            if (cndl10 > o.cndlmx) { status = 3; break; }
            if (ndf <= 0) { status = 4; break; }
        }
        double chi_add = 0.0;
        int ndf_add = 0;
        if (status == 0) {
            const float chichi = three_sigma_chi2(ndf);
            if (o.chicut >= 0.0f) {
                if (summ > (double)(o.chhuge * chichi)) status = 5;
                else if (o.chicut > 0.0f) {
                    float chlimt = o.chicut * chichi;
                    if (summ > (double)chlimt) { status = 6; chi_add = (double)chlimt; ndf_add = ndf; }
                }
            }
            if (status == 0 && o.lhuber > 1 && o.dwcut != 0.0f && resing > o.dwcut) {
                status = 6;
                chi_add = summ;
                ndf_add = ndf;
            }
        }
        if (status != 0) {
            if (tid == 0) { out.status[r] = (int8_t)status; out.chi2[r] = chi_add * dw1; out.ndf[r] = ndf_add; }
            __syncthreads();
            continue;
        }
        // ---- segments of the record's variables (group-block storage) ----
        if (o.icalcm == 1 && M.sparse && tid < 64) {
            int nseg = 0;
            for (int base = 0; base < nalg; base += 64) {
                int a = base + tid;
                int g = a < nalg ? M.group_of[gvl[a]] : -1;
                int gprev = (a > 0 && a < nalg) ? M.group_of[gvl[a - 1]] : -2;
                bool st = (a < nalg) && (a == 0 || g != gprev);
                unsigned long long m = __ballot(st);
                int s = nseg + __popcll(m & ((2ull << tid) - 1ull)) - 1;
                if (a < nalg) { segof[a] = s; if (st) segfn[s] = make_int2(M.gfirst[g], M.gfirst[g + 1] - M.gfirst[g]); }
                nseg += __popcll(m);
            }
            int npair = (nseg * nseg + nseg) / 2;
            const int64_t p0 = R.rec_pb[r];
            for (int t = tid; t < npair; t += 64) pblk[t] = t < P.max_pair ? R.pair_blk[p0 + t] : -1;
        }
        if (o.icalcm == 1)
            for (int t = tid; t < nalg * nwm; t += BNT) mask[t] = 0ull;
        __syncthreads();
        // ---- fourth loop: vector, counters, g g^T (4162-4201), support masks of G ----
        double s_chi = 0.0;
        const bool down = (o.nloopn != 1 && o.lhuber != 0);
        for (int i = tid; i < neq; i += BNT) {
            int64_t sl = R.eq_sl[e0 + i];
            uint32_t en = R.eq_n[e0 + i];
            int nl = en & 0xffff, ng = en >> 16;
            int64_t sg = sl + nl + 1;
            double rmeas = rm[i], rerr = re[i];
            double wght = 1.0 / (rerr * rerr);
            double dchi2 = wght * rmeas * rmeas;
            if (down) {
                double resid = fabs(rmeas);
                if (nter <= 3) {
                    if (resid > chuber * rerr) dchi2 = 2.0 * chuber * (resid / rerr - 0.5 * chuber);
                } else {
                    double t = resid / rerr / cauchy;
                    dchi2 = log(1.0 + t * t) * cauchy * cauchy;
                }
                wght = lw[i];
            }
            s_chi += dchi2;
            lw[i] = wght;
            for (int j = 1; j <= ng; j++) {
                double gj = bval<T>(R, sg + j);
                int pj = R.widx[sg + j];
                int vj = gv[pj];
                if (gj == 0.0) continue;
                if (vj > 0) {
                    atomicAdd(&M.vec[vj - 1], dw1 * wght * rmeas * gj);
                    atomicAdd(&M.cnt[vj - 1], 1ull);
                    if (o.icalcm == 1) {
                        int aj = gpos[pj];
                        for (int l = 1; l <= nl; l++) {
                            int kk = R.widx[sl + l] - 1;
                            atomicOr(&mask[aj * nwm + (kk >> 6)], 1ull << (kk & 63));
                        }
                        for (int k = 1; k <= j; k++) {
                            int pk_ = R.widx[sg + k];
                            int vk = gv[pk_];
                            if (vk > 0) {
                                double val = dw1 * wght * gj * bval<T>(R, sg + k);
                                int ak = gpos[pk_];
                                if (vj >= vk) band_mat_add(M, vj, vk, val, segof, segfn, pblk, aj, ak);
                                else band_mat_add(M, vk, vj, val, segof, segfn, pblk, ak, aj);
                            }
                        }
                    }
                }
            }
        }
        summ = block_sum(s_chi, red);
        if (o.icalcm == 1) {
            // ---- support classes: runs of globals with the same support of G ----
            // (one lane per global: sums over the earlier lanes give the offsets)
            if (tid < 64) {
                int ncls = 0, tot = 0, gt = 0, un = 0;
                for (int base = 0; base < nalg; base += 64) {
                    const int a = base + tid;
                    bool start = a < nalg;
                    int cnt = 0;
                    if (a < nalg) {
                        bool same = a > 0;
                        for (int w = 0; w < nwm; w++) {
                            const unsigned long long m = mask[a * nwm + w];
                            cnt += __popcll(m);
                            same = same && m == mask[(a - 1) * nwm + w];
                        }
                        start = !same;
                    }
                    const unsigned long long m = __ballot(start);
                    const int q = ncls + __popcll(m & ((2ull << tid) - 1ull)) - 1;
                    int st = start ? cnt : 0, sg = cnt, su = start ? nalg - a : 0;
                    for (int d = 1; d < 64; d <<= 1) {
                        const int x = __shfl_up(st, d, 64), y = __shfl_up(sg, d, 64), z = __shfl_up(su, d, 64);
                        if (tid >= d) { st += x; sg += y; su += z; }
                    }
                    if (a < nalg) {
                        clsof[a] = q;
                        gptr[a] = gt + sg - cnt;
                        if (start) {
                            cls0[q] = a;
                            sptr[q] = tot + st - cnt;
                            upre[q] = un + su - (nalg - a);
                        }
                    }
                    ncls += __popcll(m);
                    tot += __shfl(st, 63, 64);
                    gt += __shfl(sg, 63, 64);
                    un += __shfl(su, 63, 64);
                }
                if (tid == 0) {
                    cls0[ncls] = nalg;
                    sptr[ncls] = tot;
                    gptr[nalg] = gt;
                    upre[ncls] = un;               // work units of the Schur update: (global a, class Q <= class(a))
                    sh[5] = ncls;
                    sh[6] = tot <= P.max_sup && gt <= P.max_sup;
                }
            }
            __syncthreads();
            const int ncls = sh[5];
            if (!sh[6]) {
                if (tid == 0) { out.status[r] = 9; out.chi2[r] = 0.0; out.ndf[r] = 0; }
                __syncthreads();
                continue;
            }
            // support lists (ascending local indices) and zeroed G rows
            for (int q = tid; q < ncls; q += BNT) {
                int a = cls0[q], s = sptr[q];
                for (int w = 0; w < nwm; w++) {
                    unsigned long long m = mask[a * nwm + w];
                    while (m) {
                        int b = __ffsll((long long)m) - 1;
                        sidx[s++] = w * 64 + b + 1;
                        m &= m - 1;
                    }
                }
            }
            for (int t = tid; t < gptr[nalg]; t += BNT) gval[t] = 0.0;
            __syncthreads();
            // G = sum over equations of sqrt(dw) w g l^T, equations in order (4206-4219)
            auto slot_of = [&](int a, int kk) {
                int pos = 0;
                for (int w = 0; w < (kk >> 6); w++) pos += __popcll(mask[a * nwm + w]);
                pos += __popcll(mask[a * nwm + (kk >> 6)] & ((1ull << (kk & 63)) - 1ull));
                return &gval[gptr[a] + pos];
            };
            auto g_pairs = [&](int i, int t0, int nt) {
                const int64_t sl = R.eq_sl[e0 + i];
                const uint32_t en = R.eq_n[e0 + i];
                const int nl = en & 0xffff, ng = en >> 16;
                const int64_t sg = sl + nl + 1;
                const double wght = lw[i];
                for (int t = t0; t < ng * nl; t += nt) {
                    int j = t / nl + 1, k = t % nl + 1;
                    const int pj = R.widx[sg + j];
                    int a = gpos[pj];
                    if (a < 0) continue;
                    const int ik = R.widx[sl + k];
                    // word pairs of one equation that share the element (a label or a local
                    // index repeated in the equation) are summed by the thread of the first
                    // such pair, in the reference's (j, k) order
                    bool own = true, rep = false;
                    for (int x = 1; x <= ng; x++)
                        if (x != j && R.widx[sg + x] == pj) { rep = true; own = own && x > j; }
                    for (int x = 1; x <= nl; x++)
                        if (x != k && R.widx[sl + x] == ik) { rep = true; own = own && x > k; }
                    // zero derivatives add nothing and are not part of the support masks
                    if (!own || (!rep && bval<T>(R, sg + j) == 0.0)) continue;
                    double *ge = slot_of(a, ik - 1);
                    if (!rep) {
                        *ge = *ge + dw2 * wght * bval<T>(R, sg + j) * bval<T>(R, sl + k);
                        continue;
                    }
                    // the element exists once some pair of the run has a non-zero derivative
                    double v = 0.0;
                    bool any = false;
                    for (int j2 = j; j2 <= ng; j2++) {
                        if (R.widx[sg + j2] != pj || bval<T>(R, sg + j2) == 0.0) continue;
                        for (int k2 = k; k2 <= nl; k2++) {
                            if (R.widx[sl + k2] != ik) continue;
                            if (!any) { v = *ge; any = true; }
                            v = v + dw2 * wght * bval<T>(R, sg + j2) * bval<T>(R, sl + k2);
                        }
                    }
                    if (any) *ge = v;
                }
            };
            if (eq1 && tid < 64)
                each_equation<T>(R, e0, neq, tid, [&](int i, const EqWords<T> &E) {
                    if (E.ng == 0 || E.nl == 0) return;
                    // a label or local index that comes twice in the equation: the general form
                    bool dup = false;
                    for (int x = 1; x < E.nl; x++)
                        dup = dup || (tid > x && tid <= E.nl && E.wx == __builtin_amdgcn_readlane(E.wx, x));
                    for (int x = E.nl + 2; x < E.nl + 1 + E.ng; x++)
                        dup = dup || (tid > x && tid <= E.nl + 1 + E.ng && E.wx == __builtin_amdgcn_readlane(E.wx, x));
                    if (__any(dup)) {
                        g_pairs(i, tid, 64);
                    } else {
                        const double wght = lw[i];
                        const int div = 65536 / E.nl + 1;
                        for (int t = 0; t < E.ng * E.nl; t += 64) {
                            const int tt = min(t + tid, E.ng * E.nl - 1);
                            const int j = (tt * div) >> 16, k = tt - j * E.nl;
                            const int pg = __shfl(E.wx, E.nl + 2 + j, 64), ik = __shfl(E.wx, 1 + k, 64);
                            const double vj = lane_val(E.v, E.nl + 2 + j), vk = lane_val(E.v, 1 + k);
                            const int a = gpos[pg];
                            if (t + tid < E.ng * E.nl && a >= 0 && vj != 0.0) {
                                double *ge = slot_of(a, ik - 1);
                                *ge = *ge + dw2 * wght * vj * vk;
                            }
                        }
                    }
                    wave_order();
                });
            for (int i = 0; i < (eq1 ? 0 : neq); i++) {
                g_pairs(i, tid, BNT);
                __syncthreads();
            }
            // ---- complete inverse of the local matrix (inv = 2) into vinv ----
            // band part: columns from the right with the dbcinv recursion
            //   vs(i,j) = [i==j] W(1,i) - sum_{k=j+1}^{j+mbnd} vs(max(i,k),min(i,k)) W(1+k-j, j)
            // the mbnd columns to the right of j live in the LDS ring (slot = column mod mp1)
            const int n = nalc;
            const int nq = (mbdr * mbdr + mbdr) / 2;
            if (tid < tn) {
                for (int j = nmb; j >= 1; j--) {
                    double *colj = &ring[(j % mp1) * (NA + 1)];
                    const int kmax = min(nmb, j + mp1 - 1);
                    // off-diagonal entries of column j (rows i > j) from the columns to the right
                    for (int i = j + 1 + tid; i <= nmb; i += tn) {
                        double rxw = 0.0;
                        for (int k = j + 1; k <= kmax; k++) {
                            double vik = (k <= i) ? ring[(k % mp1) * (NA + 1) + i] : ring[(i % mp1) * (NA + 1) + k];
                            rxw = rxw - vik * vbnd[(j - 1) * mp1 + 1 + k - j];
                        }
                        colj[i] = rxw;
                        vinv[bpk64(bo + i, bo + j)] = rxw;
                    }
                    tsync();
                    if (tid == 0) {
                        double rxw = vbnd[(j - 1) * mp1 + 1];
                        for (int k = j + 1; k <= kmax; k++) rxw = rxw - colj[k] * vbnd[(j - 1) * mp1 + 1 + k - j];
                        colj[j] = rxw;
                        vinv[bpk64(bo + j, bo + j)] = rxw;
                    }
                    tsync();
                }
            }
            __threadfence_block();
            __syncthreads();
            // the border correction sum_{ib,jb} VBK(ib,jb) AUX_ib(i) AUX_jb(j)
            for (int t = tid; mbdr > 0 && t < (nmb * nmb + nmb) / 2; t += BNT) {
                int i = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f) + 1;
                while ((i * i - i) / 2 > t) i--;
                while ((i * i + i) / 2 <= t) i++;
                const int j = t - (i * i - i) / 2 + 1;
                double v = vinv[bpk64(bo + i, bo + j)];
                for (int ib = 1; ib <= mbdr; ib++)
                    for (int jb = 1; jb <= mbdr; jb++) {
                        int ij = ib > jb ? ib : jb;
                        ij = (ij * ij - ij) / 2 + (ib < jb ? ib : jb);
                        const double ai = mside == 1 ? aux[nb1 + (ib - 1) * n + i - 1] : aux[(ib - 1) * n + i];
                        const double aj = mside == 1 ? aux[nb1 + (jb - 1) * n + j - 1] : aux[(jb - 1) * n + j];
                        v = v + vbk[ij] * ai * aj;
                    }
                vinv[bpk64(bo + i, bo + j)] = v;
            }
            // border rows: -sum_jb VBK(ib,jb) AUX_jb(i) against the band, VBK within the border
            for (int t = tid; t < mbdr * nmb; t += BNT) {
                const int ib = t / nmb + 1, i = t % nmb + 1;
                double v = 0.0;
                for (int jb = 1; jb <= mbdr; jb++) {
                    int ij = ib > jb ? ib : jb;
                    ij = (ij * ij - ij) / 2 + (ib < jb ? ib : jb);
                    const double aj = mside == 1 ? aux[nb1 + (jb - 1) * n + i - 1] : aux[(jb - 1) * n + i];
                    v = v - vbk[ij] * aj;
                }
                const int dbi = mside == 1 ? ib : nmb + ib;
                vinv[bsym(dbi, bo + i)] = v;
            }
            for (int q = tid; q < nq; q += BNT) {
                int ib = 1;
                while ((ib * ib + ib) / 2 < q + 1) ib++;
                const int jb = q + 1 - (ib * ib - ib) / 2;
                const int dd = mside == 1 ? 0 : nmb;
                vinv[bpk64(dd + ib, dd + jb)] = vbk[q + 1];
            }
            __threadfence_block();
            __syncthreads();
            // ---- Schur complement: element (a >= b) -= sum_l (sum_{k in S(a)} G_ak Vinv(k,l)) G_bl ----
            const int nunit = upre[ncls];
            for (int u = tid; u < nunit; u += BNT) {
                int lo = 0, hi = ncls - 1;
                while (lo < hi) {
                    int mid = (lo + hi + 1) >> 1;
                    if (upre[mid] <= u) lo = mid; else hi = mid - 1;
                }
                const int Q = lo;
                const int a = cls0[Q] + (u - upre[Q]);
                const int ca = clsof[a];
                const int sa0 = sptr[ca], na_ = sptr[ca + 1] - sa0;
                const int sq0 = sptr[Q], nq_ = sptr[Q + 1] - sq0;
                const int bend = min(cls0[Q + 1] - 1, a);
                for (int l0 = 0; l0 < nq_; l0 += QCH) {
                    double m[QCH];
#pragma unroll
                    for (int l = 0; l < QCH; l++) m[l] = 0.0;
                    for (int s = 0; s < na_; s++) {
                        const int k = sidx[sa0 + s];
                        const double gak = gval[gptr[a] + s];
#pragma unroll
                        for (int g = 0; g < QCH; g += 4)
                            if (l0 + g < nq_) {            // four at a time (past the support: values that are not used)
#pragma unroll
                                for (int l = g; l < g + 4; l++)
                                    m[l] = m[l] + gak * vinv[bsym(k, sidx[sq0 + min(l0 + l, nq_ - 1)])];
                            }
                    }
                    for (int b = cls0[Q]; b <= bend; b++) {
                        double c = 0.0;
#pragma unroll
                        for (int l = 0; l < QCH; l++)
                            if (l0 + l < nq_) c = c + m[l] * gval[gptr[b] + l0 + l];
                        band_mat_add(M, gvl[a], gvl[b], -c, segof, segfn, pblk, a, b);
                    }
                }
            }
        }
        if (tid == 0) { out.status[r] = 0; out.chi2[r] = summ * dw1; out.ndf[r] = ndf; }
        __syncthreads();
    }
}

hipError_t launch_records_band(const DevRecords &R, const DevModel &M, const PassOpts &o, const RecOut &out,
                               const BandPlan &P, const int64_t *ids, int64_t nb, const int32_t *binfo,
                               double *scratch, int grid, hipStream_t s)
{
    if (nb <= 0) return hipSuccess;
    auto run = [&](auto kernel) {
        if (P.bytes > 65536) {
            hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, P.bytes);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(BNT), P.bytes, s, R, M, o, out, P, ids, nb, binfo, scratch);
        return hipGetLastError();
    };
    if (P.vinv_lds) return R.vf ? run(k_records_band<float, true>) : run(k_records_band<double, true>);
    return R.vf ? run(k_records_band<float, false>) : run(k_records_band<double, false>);
}

int band_lds_bytes(BandPlan &P)
{
    const size_t NA = P.nalc_max;
    size_t d = (size_t)P.max_gl + 4 * (size_t)P.max_eq + NA * P.mp1_max + 1 + (size_t)P.nbdr_max * NA + 1 +
               ((size_t)P.nbdr_max + 1) * NA + 1 + 2 * (NA + 1) + ((size_t)P.nbdr_max * P.nbdr_max + P.nbdr_max) / 2 + 1 +
               2 * ((size_t)P.nbdr_max + 1) + (size_t)P.mp1_max * (NA + 1) + P.max_sup + 8;
    P.nwm = (P.nalc_max + 63) / 64;
    size_t u64 = (size_t)P.max_var * P.nwm;
    size_t i32 = 2 * (size_t)P.max_gl + 3 * (size_t)P.max_var + 4 * ((size_t)P.max_var + 1) + P.max_sup + P.max_pair +
                 P.nbdr_max + 1 + 32;
    size_t b = d * 8 + u64 * 8 + i32 * 4;
    // the local inverse in LDS behind the rest where four workgroups still fit a CU, else in memory
    // (fewer workgroups cost more than its latency)
    P.vinv_lds = 0;
    const size_t at = (b + 7) / 8;
    if ((at + (size_t)P.vinv_stride) * 8 <= 40 * 1024) {
        P.vinv_lds = (int32_t)at;
        b = (at + (size_t)P.vinv_stride) * 8;
    }
    P.bytes = (int)b;
    return P.bytes;
}

} // namespace mpgpu
