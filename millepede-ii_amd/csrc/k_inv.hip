// Inversion of the global matrix ('method inversion'): symmetric Gauss-Jordan with pivots on the
// diagonal, as sqminl (src/mpnum.f90:230-355): at every step the unused diagonal element that is
// largest, and larger than eps times its original size, ties to the lowest index.
//
// One pivot at a time every step reads and writes the whole matrix (two launches and 16 n(n+1)/2
// bytes a step: 17 us for 1,830 rows, bound by launches and the passes over the matrix).  Here the
// pivots come in panels of 16.  Within a panel only the diagonal and the pivot columns are kept up
// to date (k_inv_panel, one workgroup: column k of the current matrix is its column at the start of
// the panel less the panel's earlier columns), so the pivot order is that of the single steps; then
// one pass applies the panel to the matrix (k_inv_update).  With K the panel's pivots, R the other
// rows, A_KK = L D L^T in pivot order and A_RK = L_R D L^T:
//     A_RR -= L_R D L_R^T,   A_RK <- A_RK A_KK^-1 = L_R L^-1,   A_KK <- -A_KK^-1.
// The matrix is held square and symmetric to the bit, so that columns are contiguous; the
// right-hand side is its last row, which is never a pivot and ends as the solution.  Matrices of up
// to INV_SMALL rows are inverted in LDS by one workgroup (k_inv_small).
// 1,830 rows: 30 -> 7.1 ms; bound by the chain of pivots (search, column, update of the
// diagonal).  From 2,048 rows on the multipliers of a panel do not fit the registers of one workgroup
// and stay in memory: 2,047 rows 8.5 ms, 2,048 30 ms (one pivot at a time 37), 5,000 158 ms (262).
#include "mpgpu_internal.h"

namespace mpgpu {

#define PB 16           // pivots of a panel
#define PT 512          // threads of the panel kernel (256 registers each: the multipliers of 4 rows)
#define INV_SMALL 128
#define UT 64           // tile of the update
#define INV_EPS 1.0e-10 // sqminl's threshold for pivots (src/mpnum.f90:251)

// square copy of the packed matrix with the right-hand side as last row and column; |diagonal|,
// used flags
__global__ void k_inv_load(int n, int ld, const double *p, const double *b, double *F, double *d, double *d0, int *used)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t tot = (int64_t)(n + 1) * (n + 2) / 2;
    if (t >= tot) return;
    int64_t i = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (i * (i + 1) / 2 > t) i--;
    while ((i + 1) * (i + 2) / 2 <= t) i++;
    const int64_t j = t - i * (i + 1) / 2;
    const double v = i < n ? p[t] : j < n ? b[j] : 0.0;
    F[i * ld + j] = v;
    F[j * ld + i] = v;
    if (i == j && i < n) {
        d[i] = v;
        d0[i] = fabs(v);
        used[i] = 0;
    }
}

struct Cand { double a; int k; };
__device__ __forceinline__ Cand better(Cand x, Cand y) { return y.a > x.a || (y.a == x.a && y.k < x.k) ? y : x; }
__device__ __forceinline__ Cand wave_best(Cand c)
{
    for (int o = 32; o > 0; o >>= 1) {
        Cand y;
        y.a = __shfl_xor(c.a, o, 64);
        y.k = __shfl_xor(c.k, o, 64);
        c = better(c, y);
    }
    return c;
}

// One panel.  Thread t has rows t, t + PT, ...; RR > 0: at most RR of them, their multipliers in
// registers (else in global memory).  info[0]: pivots of this panel, info[1]: rank so far, info[2]:
// no acceptable pivot left.  Lp, Wp: multipliers and columns [PB][ld], X: L_R L^-1 [PB][ld], Mi:
// A_KK^-1 [PB][PB], pos: place of a row among the panel's pivots (-1: none).
template <int RR>
__global__ __launch_bounds__(PT) void k_inv_panel(int n, int ld, const double *F, double *d, const double *d0, int *used, int *info,
                                                  double *Lp, double *Wp, double *X, double *Mi, int *pos)
{
    constexpr int NR = RR > 0 ? RR : 1;
    __shared__ double s_a[2][PT / 64], s_l[PB][PB], s_p[PB];
    __shared__ int s_k[2][PT / 64], s_piv[PB];
    const int tid = threadIdx.x, wave = tid >> 6;
    const double eps = INV_EPS;
    if (info[2]) {
        if (tid == 0) info[0] = 0;
        return;
    }
    double L[NR][PB], dd[NR], th[NR];
    bool fr[NR];                                       // still a candidate
    if (RR > 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int i = tid + PT * r;
            fr[r] = i < n && !used[i];
            dd[r] = i < n ? d[i] : 0.0;
            th[r] = i < n ? eps * d0[i] : 0.0;
#pragma unroll
            for (int t = 0; t < PB; t++) L[r][t] = 0.0;
        }
    }
    unsigned mine = 0;                                 // rows of this thread that are pivots (bit r)
    int np = 0;
#pragma unroll(RR > 0 ? PB : 1)
    for (int s = 0; s < PB; s++) {
        Cand c{-1.0, 0x7fffffff};
        if (RR > 0) {
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const double a = fabs(dd[r]);
                if (fr[r] && a > th[r]) c = better(c, Cand{a, tid + PT * r});
            }
        } else {
            for (int i = tid; i < n; i += PT) {
                const double a = fabs(d[i]);
                if (!used[i] && a > eps * d0[i]) c = better(c, Cand{a, i});
            }
        }
        c = wave_best(c);
        if ((tid & 63) == 0) {
            s_a[s & 1][wave] = c.a;
            s_k[s & 1][wave] = c.k;
        }
        __syncthreads();
        c = Cand{s_a[s & 1][tid & (PT / 64 - 1)], s_k[s & 1][tid & (PT / 64 - 1)]};
        for (int o = PT / 128; o > 0; o >>= 1) {
            Cand y;
            y.a = __shfl_xor(c.a, o, 64);
            y.k = __shfl_xor(c.k, o, 64);
            c = better(c, y);
        }
        const int k = __builtin_amdgcn_readfirstlane(c.k);
        if (k == 0x7fffffff) break;
        const double *col = F + (int64_t)k * ld;
        double f[NR];
        if (RR > 0) {
#pragma unroll
            for (int r = 0; r < NR; r++) f[r] = col[min(tid + PT * r, n)];
        }
        // the pivot row's multipliers and the pivot
        if (tid == k % PT) {
            if (RR > 0) {
#pragma unroll
                for (int r = 0; r < NR; r++)
                    if (r == k / PT) {
#pragma unroll
                        for (int t = 0; t < s; t++) s_l[s][t] = L[r][t];
                        s_p[s] = dd[r];
                        fr[r] = false;
                        mine |= 1u << r;
                    }
            } else {
                for (int t = 0; t < s; t++) s_l[s][t] = Lp[(int64_t)t * ld + k];
                s_p[s] = d[k];
            }
            s_piv[s] = k;
            used[k] = 1;
        }
        __syncthreads();
        const double p = s_p[s], ip = 1.0 / p;
        if (RR > 0) {
#pragma unroll
            for (int r = 0; r < NR; r++) {
                double u = f[r];
#pragma unroll
                for (int t = 0; t < s; t++) u = u - L[r][t] * (s_l[s][t] * s_p[t]);
                const int i = tid + PT * r;
                if (((mine >> r) & 1u) || i > n) u = 0.0;
                L[r][s] = u * ip;
                dd[r] = dd[r] - u * L[r][s];
                if (i <= n) {
                    Wp[(int64_t)s * ld + i] = u;
                    Lp[(int64_t)s * ld + i] = L[r][s];
                }
            }
        } else {
            for (int i = tid; i <= n; i += PT) {
                double u = col[i];
                for (int t = 0; t < s; t++) u = u - Lp[(int64_t)t * ld + i] * (s_l[s][t] * s_p[t]);
                for (int t = 0; t <= s; t++)
                    if (s_piv[t] == i) u = 0.0;
                const double l = u * ip;
                Wp[(int64_t)s * ld + i] = u;
                Lp[(int64_t)s * ld + i] = l;
                if (i < n) d[i] = d[i] - u * l;
            }
        }
        np = s + 1;
    }
    __syncthreads();
    // X = L_R L^-1: x_s = l_s - sum_{t > s} x_t L_ts
    auto solve_row = [&](int i, double (&x)[PB]) {
#pragma unroll
        for (int s = PB - 1; s >= 0; s--)
#pragma unroll
            for (int t = s + 1; t < PB; t++)
                if (t < np) x[s] = x[s] - x[t] * s_l[t][s];
        if (i > n) return;
#pragma unroll
        for (int s = 0; s < PB; s++)
            if (s < np) X[(int64_t)s * ld + i] = x[s];
        int q = -1;
        for (int s = 0; s < np; s++)
            if (s_piv[s] == i) q = s;
        pos[i] = q;
    };
    if (RR > 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int i = tid + PT * r;
            if (i < n) d[i] = dd[r];
            solve_row(i, L[r]);
        }
    } else {
        for (int i = tid; i <= n; i += PT) {
            double x[PB];
#pragma unroll
            for (int s = 0; s < PB; s++) x[s] = s < np ? Lp[(int64_t)s * ld + i] : 0.0;
            solve_row(i, x);
        }
    }
    // A_KK^-1 = L^-T D^-1 L^-1, column c per thread: L y = e_c, y / D, L^T z = y
    if (tid < np) {
        double y[PB];
#pragma unroll
        for (int s = 0; s < PB; s++) {
            y[s] = s == tid ? 1.0 : 0.0;
#pragma unroll
            for (int t = 0; t < s; t++)
                if (s < np) y[s] = y[s] - s_l[s][t] * y[t];
        }
#pragma unroll
        for (int s = 0; s < PB; s++)
            if (s < np) y[s] = y[s] / s_p[s];
#pragma unroll
        for (int s = PB - 1; s >= 0; s--) {
#pragma unroll
            for (int t = s + 1; t < PB; t++)
                if (t < np) y[s] = y[s] - s_l[t][s] * y[t];
        }
#pragma unroll
        for (int s = 0; s < PB; s++)
            if (s < np) Mi[tid * PB + s] = y[s];
    }
    if (tid == 0) {
        info[0] = np;
        info[1] += np;
        if (np < PB) info[2] = 1;
    }
}

// the panel's pass over the matrix: 64 x 64 tiles, 4 x 4 values per thread; element (i, j), i >= j:
// minus column value of row i times multiplier of row j, pivot by pivot (both triangles alike)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_inv_update(int n, int ld, double *F, const int *info, const double *Lp, const double *Wp,
                                                    const double *X, const double *Mi, const int *pos)
{
    const int np = info[0];
    if (np == 0) return;
    __shared__ double sw[2][PB][UT], sl[2][PB][UT];    // rows, columns of the tile
    const int ti = blockIdx.y, tj = blockIdx.x, t = threadIdx.x;
    const int c = t & 15, r = t >> 4;                  // columns c + 16 y, rows r + 16 x
    // the tile's values and the panel's places travel while the panel is staged
    double f[4][4];
    int pr[4], pc[4];
#pragma unroll
    for (int x = 0; x < 4; x++) {
#pragma unroll
        for (int y = 0; y < 4; y++)
            f[x][y] = F[(int64_t)min(ti * UT + r + 16 * x, n) * ld + min(tj * UT + c + 16 * y, n)];
        pr[x] = pos[min(ti * UT + r + 16 * x, n)];
        pc[x] = pos[min(tj * UT + c + 16 * x, n)];
    }
#pragma unroll
    for (int e = t; e < PB * UT; e += 256) {
        const int s = e / UT, q = e % UT;
        const int i = min(ti * UT + q, n), j = min(tj * UT + q, n);
        const bool on = s < np;
        sw[0][s][q] = on ? Wp[(int64_t)s * ld + i] : 0.0;
        sl[0][s][q] = on ? Lp[(int64_t)s * ld + i] : 0.0;
        sw[1][s][q] = on ? Wp[(int64_t)s * ld + j] : 0.0;
        sl[1][s][q] = on ? Lp[(int64_t)s * ld + j] : 0.0;
    }
    __syncthreads();
    const bool lower = ti >= tj;
    auto run = [&](const double (*a)[UT], const double (*b)[UT], double (&g)[4][4]) {
#pragma unroll 2
        for (int s = 0; s < PB; s++) {
            double u[4], v[4];
#pragma unroll
            for (int x = 0; x < 4; x++) { u[x] = a[s][r + 16 * x]; v[x] = b[s][c + 16 * x]; }
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int y = 0; y < 4; y++) g[x][y] = g[x][y] - u[x] * v[y];
        }
    };
    if (ti == tj) {
        // both forms, the one for each element's triangle kept
        double g[4][4];
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int y = 0; y < 4; y++) g[x][y] = f[x][y];
        run(sw[0], sl[1], f);
        run(sl[0], sw[1], g);
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int y = 0; y < 4; y++)
                if (r + 16 * x < c + 16 * y) f[x][y] = g[x][y];
    } else if (lower) run(sw[0], sl[1], f);
    else run(sl[0], sw[1], f);
#pragma unroll
    for (int x = 0; x < 4; x++) {
        const int i = ti * UT + r + 16 * x;
        if (i > n) continue;
        const int pi = pr[x];
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const int j = tj * UT + c + 16 * y;
            if (j > n) continue;
            const int pj = pc[y];
            double v = f[x][y];
            if (pi >= 0 && pj >= 0) v = -Mi[max(pi, pj) * PB + min(pi, pj)];
            else if (pi >= 0) v = X[(int64_t)pi * ld + j];
            else if (pj >= 0) v = X[(int64_t)pj * ld + i];
            F[(int64_t)i * ld + j] = v;
        }
    }
}

// inverse (sign turned) into the packed matrix and the solution; after a rank defect the rows and
// columns without a pivot are cleared (sqminl, src/mpnum.f90:320-331)
__global__ void k_inv_store(int n, int ld, const double *F, const int *used, const int *info, double *p, double *x)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t tot = (int64_t)n * (n + 1) / 2;
    if (t < n) x[t] = info[2] && !used[t] ? 0.0 : F[(int64_t)n * ld + t];
    if (t >= tot) return;
    int64_t i = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (i * (i + 1) / 2 > t) i--;
    while ((i + 1) * (i + 2) / 2 <= t) i++;
    const int64_t j = t - i * (i + 1) / 2;
    p[t] = info[2] && !used[i] && !used[j] ? 0.0 : -F[i * ld + j];
}

// The whole inversion in LDS, one pivot at a time: square matrix with the right-hand side as last
// row.  (Rows of n + 2 values: accesses along a row are free of bank conflicts.  Along a column or the
// diagonal, in the load and the pivot search, lanes meet in few banks where n + 2 or n + 3 is a multiple
// of 16; lengths that avoid this made the whole no faster, 204 instead of 199 us for 80 rows.)
__global__ __launch_bounds__(1024) void k_inv_small(int n, double *p, const double *b, double *x, int *info)
{
    extern __shared__ double sm[];
    const int ld = n + 2, tid = threadIdx.x, m = n + 1;
    double *A = sm;                            // [n + 1][ld]
    double *col = A + m * ld;                  // [n + 1] the pivot's column
    double *th = col + m;                      // [n]
    __shared__ double s_a[16];
    __shared__ int s_k[16];
    const double eps = INV_EPS;
    const int tot = n * (n + 1) / 2;
    for (int t = tid; t < tot; t += 1024) {
        int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
        while (i * (i + 1) / 2 > t) i--;
        while ((i + 1) * (i + 2) / 2 <= t) i++;
        const int j = t - i * (i + 1) / 2;
        const double v = p[t];
        A[i * ld + j] = v;
        A[j * ld + i] = v;
        if (i == j) th[i] = eps * fabs(v);
    }
    for (int t = tid; t < m; t += 1024) {
        const double v = t < n ? b[t] : 0.0;
        A[n * ld + t] = v;
        A[t * ld + n] = v;
    }
    __syncthreads();
    int rank = 0;
    bool stop = false, fr = tid < n;           // thread i < n: row i is a candidate
    for (int s = 0; s < n; s++) {
        Cand c{-1.0, 0x7fffffff};
        if (fr) {
            const double a = fabs(A[tid * ld + tid]);
            if (a > th[tid]) c = Cand{a, tid};
        }
        if (tid < INV_SMALL) {
            c = wave_best(c);
            if ((tid & 63) == 0) { s_a[tid >> 6] = c.a; s_k[tid >> 6] = c.k; }
        }
        __syncthreads();
        c = better(Cand{s_a[0], s_k[0]}, Cand{s_a[1], s_k[1]});
        const int k = c.k;
        if (k == 0x7fffffff) { stop = true; break; }
        rank++;
        if (tid < m) col[tid] = A[k * ld + tid];
        if (tid == k) fr = false;
        __syncthreads();
        const double vinv = 1.0 / col[k];
        for (int i = tid >> 5; i < m; i += 32)
            for (int j = tid & 31; j < m; j += 32) {
                double v;
                if (i == k && j == k) v = -vinv;
                else if (i == k) v = col[j] * vinv;
                else if (j == k) v = col[i] * vinv;
                else v = A[i * ld + j] - (col[min(i, j)] * vinv) * col[max(i, j)];
                A[i * ld + j] = v;
            }
        __syncthreads();
    }
    // candidates left after a rank defect are cleared
    if (tid < n) th[tid] = stop && fr ? 1.0 : 0.0;
    __syncthreads();
    for (int t = tid; t < tot; t += 1024) {
        int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
        while (i * (i + 1) / 2 > t) i--;
        while ((i + 1) * (i + 2) / 2 <= t) i++;
        const int j = t - i * (i + 1) / 2;
        p[t] = th[i] != 0.0 && th[j] != 0.0 ? 0.0 : -A[i * ld + j];
    }
    if (tid < n) x[tid] = th[tid] != 0.0 ? 0.0 : A[n * ld + tid];
    if (tid == 0) { info[0] = 0; info[1] = rank; info[2] = stop; }
}

__global__ void k_inv_info(int *info) { info[0] = info[1] = info[2] = 0; }

// ---------------------------------------------------------------------------------------------
// One pivot at a time in the packed matrix itself, for matrices whose square copy does not fit (from
// 135,000 rows on 288 GB, where matrix and copy take a quarter each): k_gj_pivot picks the pivot as
// the sequential scan does and stages the scaled pivot column, k_gj_update applies the elimination
// with the reference's operand order.  used[n] (0 free / 1 used), info[0] = k (1-based), info[1] =
// rank, info[2] = stop.  1,830 rows: 30 ms (panels 7.1 ms).
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ int64_t inv_pk(int64_t i, int64_t j) { return (i * i - i) / 2 + j - 1; }
__global__ void k_gj_init(int n, const double *v, double *diag, int *used, int *info)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        diag[i] = fabs(v[inv_pk(i + 1, i + 1)]);
        used[i] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) { info[0] = 0; info[1] = 0; info[2] = 0; }
}

__global__ __launch_bounds__(1024) void k_gj_pivot(int n, double *v, const double *diag, int *used, int *info,
                                                   double *vk, double *b, double eps)
{
    __shared__ double sv[1024];
    __shared__ int si[1024];
    if (info[2]) return;
    double best = -1.0;
    int bi = 0x7fffffff;
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        if (used[j]) continue;
        double a = fabs(v[inv_pk(j + 1, j + 1)]);
        if (a > eps * diag[j] && (a > best || (a == best && j < bi))) { best = a; bi = j; }
    }
    sv[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            double a = sv[threadIdx.x + o];
            int ai = si[threadIdx.x + o];
            if (a > sv[threadIdx.x] || (a == sv[threadIdx.x] && ai < si[threadIdx.x])) { sv[threadIdx.x] = a; si[threadIdx.x] = ai; }
        }
        __syncthreads();
    }
    int k = si[0];
    if (sv[0] < 0.0 || k == 0x7fffffff) { // no pivot: stop; clearing happens in k_gj_clear
        if (threadIdx.x == 0) { info[0] = 0; info[2] = 1; }
        return;
    }
    const int K = k + 1;
    const int64_t kk = inv_pk(K, K);
    const double vkk = 1.0 / v[kk];
    // scaled column k: vk(j) = v(jk)*vkk, vk(k) = 0  (sqminl lines 299-311)
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        int J = j + 1;
        if (J == K) vk[j] = 0.0;
        else {
            int64_t jk = J < K ? inv_pk(K, J) : inv_pk(J, K);
            vk[j] = v[jk] * vkk;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        used[k] = 1;
        info[0] = K;
        info[1] += 1;
        b[k] = b[k] * vkk;
        vk[n] = vkk;
    }
}

// elimination (sqminl lines 312-319): v(jl) -= vk(l) * (vk(j)/vkk) for j,l != k;
// column k takes vk, v(kk) = -vkk; b(j) -= b(k)*(vk(j)/vkk)
__global__ void k_gj_update(int n, double *v, const double *vk, double *b, const int *info)
{
    if (info[2]) return;
    const int K = info[0];
    const double vkk = vk[n];
    const int64_t total = ((int64_t)n * (n + 1)) / 2;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int64_t J = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5) + 1;
        while ((J * J - J) / 2 > t) J--;
        while ((J * J + J) / 2 <= t) J++;
        int64_t L = t - (J * J - J) / 2 + 1;
        if (J == K && L == K) v[t] = -vkk;
        else if (J == K) v[t] = vk[L - 1];
        else if (L == K) v[t] = vk[J - 1];
        else {
            double vjk = vk[J - 1] / vkk;
            v[t] = v[t] - vk[L - 1] * vjk;
        }
    }
    if (blockIdx.x == 0) {
        const double bk = b[K - 1];
        for (int j = threadIdx.x; j < n; j += blockDim.x) {
            if (j + 1 == K) continue;
            double vjk = vk[j] / vkk;
            b[j] = b[j] - bk * vjk;
        }
    }
}

// rank defect: clear rows/columns of unused pivots (sqminl lines 320-331), then negate all
__global__ void k_gj_finish(int n, double *v, double *b, const int *used, const int *info)
{
    const int64_t total = ((int64_t)n * (n + 1)) / 2;
    const bool clear = info[2] != 0;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int64_t J = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5) + 1;
        while ((J * J - J) / 2 > t) J--;
        while ((J * J + J) / 2 <= t) J++;
        int64_t L = t - (J * J - J) / 2 + 1;
        double x = v[t];
        if (clear && !used[J - 1] && !used[L - 1]) x = 0.0;
        v[t] = -x;
    }
    if (clear && blockIdx.x == 0)
        for (int j = threadIdx.x; j < n; j += blockDim.x) if (!used[j]) b[j] = 0.0;
}

static void gauss_jordan_packed(int n, double *p, const double *b, double *x, int *info, hipStream_t s)
{
    DBuf<double> diag, vk;
    DBuf<int> used;
    diag.alloc(n);
    vk.alloc(n + 1);
    used.alloc(n);
    HIPCHK(hipMemcpyAsync(x, b, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    const unsigned grid = (unsigned)std::min<int64_t>(((int64_t)n * (n + 1) / 2 + 255) / 256, 8192);
    hipLaunchKernelGGL(k_gj_init, dim3((n + 255) / 256), dim3(256), 0, s, n, p, diag.p, used.p, info);
    for (int k = 0; k < n; k++) {
        hipLaunchKernelGGL(k_gj_pivot, dim3(1), dim3(1024), 0, s, n, p, diag.p, used.p, info, vk.p, x, INV_EPS);
        hipLaunchKernelGGL(k_gj_update, dim3(grid), dim3(256), 0, s, n, p, vk.p, x, info);
    }
    hipLaunchKernelGGL(k_gj_finish, dim3(grid), dim3(256), 0, s, n, p, x, used.p, info);
    HIPCHK(hipGetLastError());
}

// packed matrix p (n rows) -> its inverse, x = inverse times b; info[1]: rank
void gauss_jordan(int n, double *p, const double *b, double *x, int *info, hipStream_t s)
{
    if (n <= INV_SMALL) {
        const int lds = ((n + 1) * (n + 2) + 2 * n + 1) * 8;
        if (lds > 65536) HIPCHK(hipFuncSetAttribute((const void *)k_inv_small, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        hipLaunchKernelGGL(k_inv_small, dim3(1), dim3(1024), lds, s, n, p, b, x, info);
        HIPCHK(hipGetLastError());
        return;
    }
    const int ld = (n + 1 + 15) / 16 * 16;
    DBuf<double> F, d, d0, Lp, Wp, X, Mi;
    DBuf<int> used, pos;
    try {
        F.alloc((size_t)(n + 1) * ld);
    } catch (const MemError &) {
        gauss_jordan_packed(n, p, b, x, info, s);
        return;
    }
    d.alloc(n);
    d0.alloc(n);
    Lp.alloc((size_t)PB * ld);
    Wp.alloc((size_t)PB * ld);
    X.alloc((size_t)PB * ld);
    Mi.alloc(PB * PB);
    used.alloc(n);
    pos.alloc(n + 1);
    hipLaunchKernelGGL(k_inv_info, dim3(1), dim3(1), 0, s, info);
    const int64_t tot = (int64_t)(n + 1) * (n + 2) / 2;
    hipLaunchKernelGGL(k_inv_load, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, n, ld, p, b, F.p, d.p, d0.p, used.p);
    const unsigned nt = (n + 1 + UT - 1) / UT;
    for (int k = 0; k < n; k += PB) {
#define INV_PANEL(RR) \
    hipLaunchKernelGGL(k_inv_panel<RR>, dim3(1), dim3(PT), 0, s, n, ld, F.p, d.p, d0.p, used.p, info, Lp.p, Wp.p, X.p, Mi.p, pos.p)
        if (n + 1 <= PT) INV_PANEL(1);
        else if (n + 1 <= 2 * PT) INV_PANEL(2);
        else if (n + 1 <= 4 * PT) INV_PANEL(4);
        else INV_PANEL(0);
#undef INV_PANEL
        hipLaunchKernelGGL(k_inv_update, dim3(nt, nt), dim3(256), 0, s, n, ld, F.p, info, Lp.p, Wp.p, X.p, Mi.p, pos.p);
    }
    hipLaunchKernelGGL(k_inv_store, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, n, ld, F.p, used.p, info, p, x);
    HIPCHK(hipGetLastError());
}

} // namespace mpgpu
