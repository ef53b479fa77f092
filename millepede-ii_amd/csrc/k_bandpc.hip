// Application of MINRES's band preconditioner (equslvs, src/mpnum.f90:2600-2680: band factor of the
// parameter block, constraint block) for bands of up to 9 rows and up to 128 constraints.
//
// The band recurrences of lltfwd / lltbwd are split on two levels.  Sub-chunks of 16 rows have
// their dense inverse stored (the backward solve of a sub-chunk is the transpose of the forward
// one), so their solution with a zero boundary is 16 multiply-adds per row instead of a chain over
// the rows; the w = mbandw-1 boundary values are carried over the 16 sub-chunks of a chunk by one
// wavefront, and from chunk to chunk by the scan of k_spk_scan.  The recurrences are linear, so
// this holds for rows that lltdec has reset too.
//
// What the old chain cost: one lane walked the 256 rows of a chunk, 60 ns a row (20 us per sweep,
// two per iteration, on 24,000 parameters; 6 us now).  The forward correction by the
// carried boundary, the constraint block and the backward solve share one kernel, the constraint
// factor's inverse (m x m, formed once per matrix) replaces its two substitutions (20 us for 60
// constraints), and the backward correction is left to the kernel that takes MINRES's dot product.
//
// Contexts with eliminated constraints keep the substitutions of k_spk_*: their solves may end at the
// iteration limit, where another order of sums shows in the result (mpgpu_ctx::elim).
#include "mpgpu_internal.h"

namespace mpgpu {

#define SUB 16          // rows of a sub-chunk
#define CH 256          // rows of a chunk (spk_chunk_rows)
#define NSUB (CH / SUB)

// factor element (k, j), 1-based, zero outside the band row
__device__ __forceinline__ double band_c(const double *c, const int *india, int k, int j)
{
    const int e = india[k - 1], len = e - (k > 1 ? india[k - 2] : 0);
    return j >= k - len + 1 && j <= k ? c[e - k + j - 1] : 0.0;
}

// Thread (sub, i): i < 16 column i of the sub-chunk's inverse, into F (column-major) and B
// (row-major); then w forward and w backward responses of the rows to a unit boundary value.
template <int W>
__global__ __launch_bounds__(64) void k_bp_sub(int n, const double *c, const int *india, double *F, double *B, double *Sf,
                                               double *Sb)
{
    constexpr int NT = SUB + 2 * W;
    const int t = blockIdx.x * 64 + threadIdx.x;
    const int u = t / NT, i = t - u * NT;
    const int k0 = u * SUB + 1;
    if (k0 > n) return;
    const int k1 = min(n, k0 + SUB - 1);
    double x[SUB];
    if (i < SUB) {
        for (int r = 0; r < SUB; r++) {
            double s = r == i ? 1.0 : 0.0;
            const int k = k0 + r;
            if (r < i || k > k1) s = 0.0;
            else {
                for (int o = 1; o <= W; o++)
                    if (r - o >= i) s -= band_c(c, india, k, k - o) * x[r - o];
                s *= band_c(c, india, k, k);
            }
            x[r] = s;
            F[((size_t)u * SUB + i) * SUB + r] = s;
            B[((size_t)u * SUB + r) * SUB + i] = s;
        }
    } else if (i < SUB + W) {
        const int q = i - SUB;
        for (int k = k0; k <= k1; k++) {
            const int r = k - k0;
            double s = 0.0;
            for (int o = 1; o <= W && o < k; o++) {
                const double xi = r - o >= 0 ? x[r - o] : W + r - o == q ? 1.0 : 0.0;
                s -= band_c(c, india, k, k - o) * xi;
            }
            x[r] = s * band_c(c, india, k, k);
            Sf[(size_t)(k - 1) * W + q] = x[r];
        }
    } else {
        const int q = i - SUB - W;
        for (int k = k1; k >= k0; k--) {
            double s = 0.0;
            for (int o = 1; o <= W && k + o <= n; o++) {
                const int j = k + o;
                const double xj = j <= k1 ? x[j - k0] : j - k1 - 1 == q ? 1.0 : 0.0;
                s -= band_c(c, india, j, k) * xj;
            }
            x[k - k0] = s * band_c(c, india, k, k);
            Sb[(size_t)(k - 1) * W + q] = x[k - k0];
        }
    }
}

// responses of a chunk's rows to its own boundary, composed from those of its sub-chunks
template <int W>
__global__ __launch_bounds__(CH) void k_bp_chunk(int n, const double *Sf, const double *Sb, double *Cf, double *Cb)
{
    __shared__ double sf[CH * W], sb[CH * W], su[NSUB][W][W];
    const int r = threadIdx.x, k = blockIdx.x * CH + r;
    for (int q = 0; q < W; q++) {
        sf[r * W + q] = k < n ? Sf[(size_t)k * W + q] : 0.0;
        sb[r * W + q] = k < n ? Sb[(size_t)k * W + q] : 0.0;
    }
    for (int dir = 0; dir < 2; dir++) {
        const double *S = dir == 0 ? sf : sb;
        __syncthreads();
        if (r < W) {
            double s[W];
            for (int p = 0; p < W; p++) s[p] = p == r ? 1.0 : 0.0;
            for (int v = 0; v < NSUB; v++) {
                const int u = dir == 0 ? v : NSUB - 1 - v;
                double y[W];
                for (int p = 0; p < W; p++) su[u][r][p] = s[p];
                for (int p = 0; p < W; p++) {
                    const int row = u * SUB + (dir == 0 ? SUB - W + p : p);
                    y[p] = 0.0;
                    for (int q = 0; q < W; q++) y[p] += S[row * W + q] * s[q];
                }
                for (int p = 0; p < W; p++) s[p] = y[p];
            }
        }
        __syncthreads();
        if (k < n)
            for (int q = 0; q < W; q++) {
                double v = 0.0;
                for (int p = 0; p < W; p++) v += S[r * W + p] * su[r / SUB][q][p];
                (dir == 0 ? Cf : Cb)[(size_t)k * W + q] = v;
            }
    }
}

// inverse of the constraint block from its factor (lltdec's form, full rows), one column per
// wavefront, two rows per lane
__global__ __launch_bounds__(64) void k_bp_hinv(int m, const double *h, double *hinv)
{
    extern __shared__ double sh[];
    const int lane = threadIdx.x, nh = (m * m + m) / 2;
    for (int t = lane; t < nh; t += 64) sh[t] = h[t];
    __syncthreads();
    auto H = [&](int k, int j) { return sh[(k * k + k) / 2 + j]; };   // 0-based, j <= k
    double x[2];
    for (int v = 0; v < 2; v++) x[v] = lane + 64 * v == (int)blockIdx.x ? 1.0 : 0.0;
    for (int j = 0; j < m; j++) {
        const double d = H(j, j);
        if (lane == (j & 63)) x[j >> 6] *= d;
        const double xj = __shfl(j >= 64 ? x[1] : x[0], j & 63, 64);
        for (int v = 0; v < 2; v++) {
            const int k = lane + 64 * v;
            if (k > j && k < m) x[v] -= H(k, j) * xj;
        }
    }
    for (int k = m - 1; k >= 0; k--) {
        const double d = H(k, k);
        if (lane == (k & 63)) x[k >> 6] *= d;
        const double xk = __shfl(k >= 64 ? x[1] : x[0], k & 63, 64);
        for (int v = 0; v < 2; v++) {
            const int j = lane + 64 * v;
            if (j < k) x[v] -= H(k, j) * xk;
        }
    }
    for (int v = 0; v < 2; v++) {
        const int k = lane + 64 * v;
        if (k < m) hinv[(size_t)blockIdx.x * m + k] = x[v];
    }
}


// Solution of a chunk with a zero boundary, one thread per row (b: its right-hand side): the
// sub-chunk's inverse (M), then the boundary values carried over the sub-chunks by the first
// wavefront, lane i boundary value i.  DIR 0 forward, 1 backward.
template <int W, int DIR>
__device__ __forceinline__ double bp_solve(double b, bool live, const double *M, const double (&S)[W], double *sv, double *sB,
                                           double *sS)
{
    const int r = threadIdx.x, u = r / SUB, i = r % SUB;
    sv[r] = b;
    // boundary rows of each sub-chunk: the last W (forward) or first W (backward)
    const int bi = DIR == 0 ? i - (SUB - W) : i;
    if (bi >= 0 && bi < W) {
#pragma unroll
        for (int q = 0; q < W; q++) sB[(u * W + bi) * W + q] = S[q];
    }
    __syncthreads();
    double y = 0.0;
    if (live) {
        double m[SUB];
#pragma unroll
        for (int j = 0; j < SUB; j++) m[j] = M[j * SUB];
#pragma unroll
        for (int j = 0; j < SUB; j++) y += m[j] * sv[u * SUB + j];
    }
    __syncthreads();
    sv[r] = y;
    __syncthreads();
    if (r < 64) {
        const int l = r < W ? r : 0;
        double s = 0.0;
        for (int v = 0; v < NSUB; v++) {
            const int w = DIR == 0 ? v : NSUB - 1 - v;
            if (r < W) sS[w * W + r] = s;
            double t = sv[w * SUB + (DIR == 0 ? SUB - W + l : l)];
#pragma unroll
            for (int q = 0; q < W; q++) t += sB[(w * W + l) * W + q] * wave_lane(s, q);
            s = t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < W; q++) y += S[q] * sS[u * W + q];
    return y;
}

// forward: y = chunk-local solution for the right-hand side x
template <int W>
__global__ __launch_bounds__(CH) void k_bp_fwd(int n, const double *x, const double *F, const double *Sf, double *y)
{
    __shared__ double sv[CH], sB[NSUB * W * W], sS[NSUB * W];
    const int r = threadIdx.x, k = blockIdx.x * CH + r;
    const bool live = k < n;
    double S[W];
#pragma unroll
    for (int q = 0; q < W; q++) S[q] = live ? Sf[(size_t)k * W + q] : 0.0;
    const double v = bp_solve<W, 0>(live ? x[k] : 0.0, live, F + (size_t)(k / SUB) * SUB * SUB + k % SUB, S, sv, sB, sS);
    if (live) y[k] = v;
}

// value of row i after the forward sweep: its chunk-local solution corrected by the carried boundary
template <int W>
__device__ __forceinline__ double bp_fixed(int i, const double *y, const double *C, const double *t)
{
    double v = y[i];
    const int ch = i / CH;
    if (ch > 0) {
#pragma unroll
        for (int q = 0; q < W; q++) v += C[(size_t)i * W + q] * t[(size_t)ch * W + q];
    }
    return v;
}

// d_j = x[n+j] - K_j . y, y corrected
template <int W>
__global__ __launch_bounds__(256) void k_bp_cdot(int n, const int *cb, const int64_t *koff, const double *kmat, const double *x,
                                                 const double *y, const double *Cf, const double *t, double *d)
{
    __shared__ double red[4];
    const int j = blockIdx.x, i0 = cb[2 * j], in = min(cb[2 * j + 1], n - i0);
    const double *kj = kmat + koff[j];
    double acc = 0.0;
    for (int i = threadIdx.x; i < in; i += 256) acc += kj[i] * bp_fixed<W>(i0 + i, y, Cf, t);
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) d[j] = x[n + j] - ((red[0] + red[1]) + (red[2] + red[3]));
}

// Constraint block (lambda = -H^-1 d, y -= K^T lambda) and chunk-local backward solution, in place.
// Every workgroup forms all multipliers (m^2 products from L2) and keeps the constraints whose
// range meets its rows, in ascending order.
template <int W>
__global__ __launch_bounds__(CH) void k_bp_bwd(int n, int m, double *y, const double *Cf, const double *t, const double *hinv,
                                               const double *d, const int *cb, const int64_t *koff, const double *kmat,
                                               const double *B, const double *Sb)
{
    __shared__ double sv[CH], sB[NSUB * W * W], sS[NSUB * W], sl[128];
    __shared__ int s0[128], sn[128];
    __shared__ int64_t so[128];
    __shared__ int ord[128], wc[2], cnt;
    const int r = threadIdx.x, k = blockIdx.x * CH + r, k0 = blockIdx.x * CH;
    const bool live = k < n;
    double S[W];
#pragma unroll
    for (int q = 0; q < W; q++) S[q] = live ? Sb[(size_t)k * W + q] : 0.0;
    double b = live ? bp_fixed<W>(k, y, Cf, t) : 0.0;
    if (m > 0) {
        const int parts = CH / m, p = r / m, j = r - p * m;
        double l = 0.0;
        if (p < parts)
            for (int i = p; i < m; i += parts) l += hinv[(size_t)i * m + j] * d[i];
        sv[r] = l;
        bool meets = false;
        if (r < m) {
            s0[r] = cb[2 * r];
            sn[r] = cb[2 * r + 1];
            so[r] = koff[r];
            meets = s0[r] < k0 + CH && s0[r] + sn[r] > k0;
        }
        const unsigned long long bal = __ballot(meets);
        if (r < 128 && (r & 63) == 0) wc[r >> 6] = __popcll(bal);
        __syncthreads();
        if (r < m) {
            double v = 0.0;
            for (int q = 0; q < parts; q++) v += sv[q * m + r];
            sl[r] = -v;
            if (blockIdx.x == 0) y[n + r] = -v;
        }
        if (meets) ord[(r >= 64 ? wc[0] : 0) + __popcll(bal & ((1ull << (r & 63)) - 1ull))] = r;
        if (r == 0) cnt = wc[0] + (m > 64 ? wc[1] : 0);
        __syncthreads();
        if (live)
            for (int q = 0; q < cnt; q++) {
                const int c = ord[q];
                if (k >= s0[c] && k < s0[c] + sn[c]) b = b - kmat[so[c] + (k - s0[c])] * sl[c];
            }
        __syncthreads();
    }
    const double v = bp_solve<W, 1>(b, live, B + (size_t)(k / SUB) * SUB * SUB + k % SUB, S, sv, sB, sS);
    if (live) y[k] = v;
}

// the correction of the backward sweep by itself (the first application, MINRES-QLP)
template <int W>
__global__ __launch_bounds__(256) void k_bp_fix(int n, int nch, double *y, const double *Cb, const double *t)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n || i / CH == nch - 1) return;
    double v = y[i];
#pragma unroll
    for (int q = 0; q < W; q++) v += Cb[(size_t)i * W + q] * t[(size_t)(i / CH) * W + q];
    y[i] = v;
}

#define BP_W(w, F)                                                                                                  \
    switch (w) {                                                                                                    \
    case 1: F(1); break;                                                                                            \
    case 2: F(2); break;                                                                                            \
    case 3: F(3); break;                                                                                            \
    case 4: F(4); break;                                                                                            \
    case 5: F(5); break;                                                                                            \
    case 6: F(6); break;                                                                                            \
    case 7: F(7); break;                                                                                            \
    default: F(8); break;                                                                                           \
    }

bool bp_usable(int n, int m, int w)
{
    const int nch = (n + CH - 1) / CH;
    return spk_chunk_rows() == CH && n > 0 && w >= 1 && w <= 8 && m <= 128 && (nch == 1 || spk_scan_levels(n, w) > 0);
}
int64_t bp_sub_elems(int n) { return (int64_t)((n + SUB - 1) / SUB) * SUB * SUB; }

void l_bp_build(int n, int m, int w, const double *c, const int *india, const double *h, double *F, double *B, double *Sf,
                double *Sb, double *Cf, double *Cb, double *hinv, hipStream_t s)
{
    const int nsub = (n + SUB - 1) / SUB, nch = (n + CH - 1) / CH;
#define BP_F(W_)                                                                                                    \
    hipLaunchKernelGGL(k_bp_sub<W_>, dim3((unsigned)(((int64_t)nsub * (SUB + 2 * W_) + 63) / 64)), dim3(64), 0, s, n, c, india, F, \
                       B, Sf, Sb);                                                                                  \
    hipLaunchKernelGGL(k_bp_chunk<W_>, dim3(nch), dim3(CH), 0, s, n, Sf, Sb, Cf, Cb)
    BP_W(w, BP_F)
#undef BP_F
    if (m > 0) {
        const int lds = (m * m + m) / 2 * 8;
        if (lds > 65536) HIPCHK(hipFuncSetAttribute((const void *)k_bp_hinv, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        hipLaunchKernelGGL(k_bp_hinv, dim3(m), dim3(64), lds, s, m, h, hinv);
    }
    HIPCHK(hipGetLastError());
}

// y = M^-1 x up to the backward correction (t: the carried boundary values), which the caller's next
// kernel or l_bp_fix adds
void l_bp_apply(int n, int m, int w, const double *x, double *y, const BandPc &P, hipStream_t s)
{
    const int nch = (n + CH - 1) / CH;
#define BP_F(W_)                                                                                                    \
    hipLaunchKernelGGL(k_bp_fwd<W_>, dim3(nch), dim3(CH), 0, s, n, x, P.F, P.Sf, y);                                \
    if (nch > 1) l_spk_scan(n, W_, y, P.Af, P.nlev, P.t, 0, s);                                                     \
    if (m > 0) hipLaunchKernelGGL(k_bp_cdot<W_>, dim3(m), dim3(256), 0, s, n, P.cb, P.koff, P.kmat, x, y, P.Cf, P.t, P.d); \
    hipLaunchKernelGGL(k_bp_bwd<W_>, dim3(nch), dim3(CH), 0, s, n, m, y, P.Cf, P.t, P.hinv, P.d, P.cb, P.koff, P.kmat, P.B, P.Sb); \
    if (nch > 1) l_spk_scan(n, W_, y, P.Ab, P.nlev, P.t, 1, s)
    BP_W(w, BP_F)
#undef BP_F
}
void l_bp_fix(int n, int w, double *y, const BandPc &P, hipStream_t s)
{
    const int nch = (n + CH - 1) / CH;
    if (nch < 2) return;
#define BP_F(W_) hipLaunchKernelGGL(k_bp_fix<W_>, dim3((n + 255) / 256), dim3(256), 0, s, n, nch, y, P.Cb, P.t)
    BP_W(w, BP_F)
#undef BP_F
}

} // namespace mpgpu
