// Host-side internals of libmpgpu (not part of the C-ABI).
#pragma once
#include "mpgpu_device.h"
#include "../../include/mpgpu.h"
#include <algorithm>
#include <functional>
#include <string>
#include <unordered_map>
#include <vector>
#include <cstring>
#include <utility>

namespace mpgpu {

#define HIPCHK(x)                                                                                   \
    do {                                                                                            \
        hipError_t e_ = (x);                                                                        \
        if (e_ != hipSuccess) throw MpError(30, std::string("HIP error: ") + hipGetErrorString(e_) + \
                                                    " at " + __FILE__ + ":" + std::to_string(__LINE__)); \
    } while (0)

struct MpError {
    int code;
    std::string msg;
    MpError(int c, std::string m) : code(c), msg(std::move(m)) {}
};
// no device memory (DevCache::get)
struct MemError : MpError {
    using MpError::MpError;
};

// Device memory of a context.  Buffers made during a library call are ordered on the context's
// stream, so a freed block can serve the next buffer of that context at once; when the context ends
// (its stream has finished) its free blocks go to a store shared by the contexts of the device.
// hipFreeAsync takes 8 us for a small block and over 100 us from 1 MB on, and a job of the serving
// engine frees some two hundred.  Blocks above CACHE_BLOCK go straight to hipMallocAsync /
// hipFreeAsync, in their own size; a context keeps at most CACHE_CONTEXT bytes of free blocks and the
// store CACHE_STORE, and both are given back when an allocation fails.
class DevCache {
  public:
    DevCache(hipStream_t st, int dev);
    ~DevCache();                             // the stream has finished
    DevCache(const DevCache &) = delete;
    DevCache &operator=(const DevCache &) = delete;
    void *get(size_t bytes);
    void put(void *p, size_t bytes) noexcept;
    hipStream_t stream() const { return s; }
    size_t live() const { return live_; }    // bytes in use, their maximum, and bytes of free blocks
    size_t peak() const { return peak_; }
    size_t kept() const { return held; }
    int64_t room() const;                    // bytes new buffers may take: free on the device, within the limit
    void read_limit();                       // MPGPU_MEMORY_LIMIT_MB
    void set_share(size_t b) { share = b; }  // no more free blocks than fit below b bytes with those in use
    std::function<void()> reclaim;           // gives back what the context can do without, when an allocation fails

  private:
    hipStream_t s;
    int device;
    size_t held = 0, live_ = 0, peak_ = 0;
    size_t limit = 0;                        // most bytes in use (0: the device's)
    size_t share = SIZE_MAX;
    std::unordered_map<size_t, std::vector<void *>> free_;
    void drop();
    hipError_t fresh(void **p, size_t c);
};
size_t dev_store_kept();                     // bytes of free blocks of ended contexts
void dev_store_trim(int device, size_t most, hipStream_t st);   // frees blocks of a device until at most that many are kept
// memory of the library call in progress on this thread (none: hipMalloc / hipFree)
inline DevCache *&alloc_cache()
{
    static thread_local DevCache *c = nullptr;
    return c;
}
struct AllocScope {
    DevCache *prev;
    explicit AllocScope(DevCache *c) : prev(alloc_cache()) { alloc_cache() = c; }
    ~AllocScope() { alloc_cache() = prev; }
    AllocScope(const AllocScope &) = delete;
    AllocScope &operator=(const AllocScope &) = delete;
};

// owning device buffer; freed in the order of the stream it was made for (see DevCache)
template <typename T> struct DBuf {
    T *p = nullptr;
    size_t n = 0;
    DevCache *as = nullptr;
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { release(); }
    void release()
    {
        if (p) {
            if (as) as->put(p, sizeof(T) * n);
            else (void)hipFree(p);
        }
        p = nullptr;
        n = 0;
        as = nullptr;
    }
    void alloc(size_t count)
    {
        if (count == n && p) return;
        release();
        if (count == 0) return;
        as = alloc_cache();
        if (as) p = (T *)as->get(sizeof(T) * count);
        else HIPCHK(hipMalloc((void **)&p, sizeof(T) * count));
        n = count;
    }
    void upload(const T *h, size_t count, hipStream_t s)
    {
        alloc(count);
        if (count) HIPCHK(hipMemcpyAsync(p, h, sizeof(T) * count, hipMemcpyHostToDevice, s));
    }
    void upload(const std::vector<T> &v, hipStream_t s) { upload(v.data(), v.size(), s); }
    void download(T *h, size_t count, hipStream_t s) const
    {
        if (count) HIPCHK(hipMemcpyAsync(h, p, sizeof(T) * count, hipMemcpyDeviceToHost, s));
    }
    void zero(hipStream_t s)
    {
        if (n) HIPCHK(hipMemsetAsync(p, 0, sizeof(T) * n, s));
    }
    void swap(DBuf &o)
    {
        std::swap(p, o.p);
        std::swap(n, o.n);
        std::swap(as, o.as);
    }
};

// HIP events that live until the end of the enclosing scope
struct EventPool {
    std::vector<hipEvent_t> ev;
    EventPool() = default;
    EventPool(const EventPool &) = delete;
    EventPool &operator=(const EventPool &) = delete;
    ~EventPool()
    {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    }
    hipEvent_t get()
    {
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        ev.push_back(e);
        return e;
    }
};

struct EqBlock {
    int kind; // 0 constraint, 1 measurement
    double rhs, sigma;
    std::vector<int32_t> labels;
    std::vector<double> factors;
};

// kernels (k_records.hip, k_solve.hip, k_chol.hip)
hipError_t launch_records(const DevRecords &R, const DevModel &M, const PassOpts &o, const RecOut &out, const LdsPlan &P,
                          int64_t rec_begin, int64_t rec_end, int grid, hipStream_t s, const MonCtx &mon);
int lds_bytes(LdsPlan &P);
hipError_t launch_block_gather(int64_t nblock, const int64_t *boff, const int32_t *brg, const int32_t *bcol,
                               const int32_t *gfirst, const int64_t *ptr, const int64_t *src, const double *cbuf,
                               double *mat, double *vec, hipStream_t s);
hipError_t launch_records_band(const DevRecords &R, const DevModel &M, const PassOpts &o, const RecOut &out,
                               const BandPlan &P, const int64_t *ids, int64_t nb, const int32_t *binfo,
                               double *scratch, int grid, hipStream_t s);
int band_lds_bytes(BandPlan &P);
void l_mupdat(const DevModel &M, int32_t n, const int32_t *i, const int32_t *j, const double *v, hipStream_t s);
void l_get_diag(const DevModel &M, int32_t n, double *d, hipStream_t s);
void l_get_band(const DevModel &M, int32_t n, int32_t mbandw, const int32_t *india, double *c, hipStream_t s);
void l_dot(int64_t n, const double *a, const double *b, double *part, double *out, hipStream_t s);
void l_pass_stats(int64_t n, const double *chi2, const int32_t *ndf, const int8_t *st, double *part, long long *ndfsum,
                  unsigned long long *hist, double *chi_out, hipStream_t s);
// inversion of the packed matrix p in place and x = A^-1 b; info[1]: rank (k_inv.hip)
void gauss_jordan(int n, double *p, const double *b, double *x, int *info, hipStream_t s);
// y = A x for the packed symmetric matrix; scratch: packed_symv_scratch(n) doubles
void l_packed_symv(int n, const double *a, const double *x, double *y, double *scratch, hipStream_t s);
int64_t packed_symv_scratch(int n);
// the same product with the partial sums in a fixed file-scope device array (no allocation);
// n <= noalloc_max_n()
hipError_t noalloc_packed_symv(int device, int n, const double *a, const double *x, double *y, hipStream_t s);
int noalloc_max_n();
void l_mr_scale(int64_t n, const MrState *st, const double *y, double *v, hipStream_t s);
void l_mr_mid(int64_t n, MrState *st, int first, const double *v, const double *r1, double *y, double *part, hipStream_t s);
void l_mr_sub(int64_t n, const MrState *st, const double *r2, double *r1, double *y, int keep, hipStream_t s);
void l_mr_end(int64_t n, MrState *st, const double *r2, double *y, int w, int nb, const double *Cb, const double *t, double *part,
              hipStream_t s);
void l_mr_next(int64_t n, const MrState *st, const double *y, double *v, double *w, double *w2, double *x, hipStream_t s);
// A part of a block row for the block product: n off-diagonal blocks from block b0 of the values at
// a[off], and with diag the row's diagonal block behind them (ga < 0: no part).  The parts of a row
// are summed by the columns pass, so the split is part of the sum's order and every variant of the
// product uses the same one.
struct RowPart {
    int32_t ga, b0, n, diag;
    int64_t off;
};
struct BlockParts {
    int64_t n = 0;                  // entries of part (the last ones may be empty)
    const RowPart *part = nullptr;
    const int64_t *ptr = nullptr;   // per block row: its first part
    double *yp = nullptr;           // 8 sums per part
};
void l_block_symv(int32_t ngroup, const int64_t *brow, const int32_t *bcf, const int64_t *boff, const int32_t *gfirst,
                  const int64_t *ccol_ptr, const int64_t *cc_off, const int32_t *cc_fn, const double *a,
                  const double *x, double *y, int32_t nvar, int64_t nall, int32_t maxgrp, const int32_t *cc_blk,
                  double *tb, int32_t ugrp, const int32_t *bcol, int64_t nblock, const BlockParts &parts, int variant,
                  hipStream_t s);
// variants of the product with identical arithmetic (for the autotuner); returns their number
int block_symv_variants(int32_t ugrp, int32_t maxgrp, int *out);
void l_cons_symv(int32_t ncon, int32_t nvar, const int64_t *cptr, const int32_t *cidx, const double *cval, const double *x,
                 double *y, hipStream_t s);
void l_scale_copy(int64_t n, double sc, const double *a, double *o, hipStream_t s);
void l_axpy_neg(int64_t n, double c, const double *r, double *y, hipStream_t s);
void l_minres_update(int64_t n, const double *v, double *w, double *w1, double *w2, double *x, double oldeps, double delta,
                     double denom, double phi, hipStream_t s);
void l_qlp_minres(int64_t n, const double *v, double *w, double *wl, double *wl2, double *x, double epln, double dlta,
                  double sc, double tau, int upd_w, int upd_x, hipStream_t s);
void l_qlp_step(int64_t n, double *v, double *w, double *wl, double *wl2, double *x, double *xl2, const QlpStep &c,
                hipStream_t s);
void l_copy(int64_t n, const double *a, double *b, hipStream_t s);
void l_xpby(int64_t n, const double *z, double beta, double *p, hipStream_t s);
void l_sub(int64_t n, const double *b, const double *ax, double *r, hipStream_t s);
void l_precons(int32_t n, int32_t p, const double *diag, double *cu, int *nrkd, const int64_t *cptr, const int32_t *cidx,
               const double *cval, double *sm, double *scratch, hipStream_t s);
void l_presols(int32_t n, int32_t p, const double *cu, const int64_t *cptr, const int32_t *cidx, const double *cval,
               const double *sm, const double *y, double *x, hipStream_t s);
void l_lltdec(int n, double *c, const int *india, int *nrkd, int iopt, int mbw, hipStream_t s);
// the band factorization by chunks of rows in parallel, with the sequential result bit for bit
// (falls back to the sequential kernel when a chunk does not catch up); L: n * mbw doubles,
// bad: n bytes, flag: three ints of device scratch
bool lltdec_parallel(int n, int mbw);
void l_lltdec_par(int n, double *c, const int *india, int *nrkd, int iopt, int mbw, double *L, int8_t *bad, int *flag,
                  hipStream_t s);
void l_band_k(int32_t ncon, int n, const double *c, const int *india, const int *cb, const int64_t *koff, double *kmat,
              int mbw, hipStream_t s);
void l_band_h(int32_t m, const int *cb, const int64_t *koff, const double *kmat, double *h, const int *hind, int *nrkd2,
              hipStream_t s);
void l_equslvs(int n, int m, const double *c, const int *india, const int *cb, const int64_t *koff, const double *kmat,
               const double *h, const int *hind, double *x, hipStream_t s);

void l_spk_build(int n, int w, const double *c, const int *india, double *Sf, double *Sb, double *scr, hipStream_t s);
void l_equslvs_spike(int n, int m, int w, const double *c, const int *india, const double *Sf, const double *Sb,
                     double *tbuf, const int *cb, const int64_t *koff, const double *kmat, const double *h, const int *hind,
                     double *dtmp, double *x, const double *Af, const double *Ab, int nlev, hipStream_t s);
int spk_chunk_rows();   // rows per chunk of the chunk-parallel band solves
int spk_scan_levels(int n, int w);
void l_spk_scan_build(int n, int w, const double *Sf, const double *Sb, double *Af, double *Ab, int nlev, hipStream_t s);

void l_spk_scan(int n, int w, const double *x, const double *A, int nlev, double *t, int backward, hipStream_t s);
// application of the band preconditioner (k_bandpc.hip): sub-chunk inverses, responses of the rows
// to the boundaries of their sub-chunk (S) and chunk (C), scan levels (A), carried boundary values
// (t), inverse of the constraint block and its right-hand side
struct BandPc {
    const double *F, *B, *Sf, *Sb, *Cf, *Cb, *Af, *Ab, *hinv, *kmat;
    const int *cb;
    const int64_t *koff;
    double *t, *d;
    int nlev;
};
bool bp_usable(int n, int m, int w);
int64_t bp_sub_elems(int n);
void l_bp_build(int n, int m, int w, const double *c, const int *india, const double *h, double *F, double *B, double *Sf,
                double *Sb, double *Cf, double *Cb, double *hinv, hipStream_t s);
void l_bp_apply(int n, int m, int w, const double *x, double *y, const BandPc &P, hipStream_t s);
void l_bp_fix(int n, int w, double *y, const BandPc &P, hipStream_t s);

// dense LDL^T (k_chol.hip): full column-major n x n matrix (lda = n), lower triangle.  The
// factor keeps the raw pivots on the diagonal, w_i = 1/d_i (d_i > 0) or d_i in w, and needs
// ldl_work_elems(n) elements of work (panel buffer and the inverse diagonal blocks, used again
// by the solves).
int64_t ldl_work_elems(int n);
hipError_t ldl_factor(int n, double *a, int lda, double *w, double *work, hipStream_t s);
hipError_t ldl_factor32(int n, float *a, int lda, float *w, float *work, hipStream_t s);
void ldl_solve(int n, const double *a, int lda, const double *w, const double *work, double *x, int nrhs, int64_t ldx,
               hipStream_t s);
void ldl_solve32(int n, const float *a, int lda, const float *w, const float *work, double *x, int nrhs, int64_t ldx,
                 hipStream_t s);
void ldl_pivots(int n, const double *a, int lda, double *d, hipStream_t s);
void ldl_pivots32(int n, const float *a, int lda, double *d, hipStream_t s);
// diagonal of A^-1 from the FP64 factor (in the factor's index order); e: scratch of n * nbk
void ldl_inv_diag(int n, const double *a, int lda, const double *w, const double *work, double *e, int nbk, double *d,
                  hipStream_t s);
void l_reverse(int n, double *x, int nrhs, int64_t ldx, hipStream_t s);
void l_packed_to_full(int n, const double *packed, double *full, int lda, int rev, hipStream_t s);
// sc (may be NULL): symmetric scaling, element (i, j) multiplied by sc[i] sc[j]
void l_packed_to_full32(int n, const double *packed, float *full, int lda, int rev, const double *sc, hipStream_t s);
void l_scale_cols(int n, const double *d, double *x, int nrhs, int64_t ldx, hipStream_t s);
void l_add_cct(int32_t ncon, const int64_t *cptr, const int32_t *cidx, const double *cval, double rho, double *a,
               int lda, int n, int rev, hipStream_t s);
void l_add_cct32(int32_t ncon, const int64_t *cptr, const int32_t *cidx, const double *cval, double rho, float *a,
                 int lda, int n, int rev, const double *sc, hipStream_t s);
void l_cct_apply(int32_t ncon, const int64_t *cptr, const int32_t *cidx, const double *cval, double rho,
                 const double *x, double *y, hipStream_t s);
void l_col_dots(int n, int nrhs, const double *a, const double *b, double *out, hipStream_t s);
void l_col_axpy(int n, int nrhs, const double *alpha, double sg, const double *x, double *y, hipStream_t s);
void l_col_xpby(int n, int nrhs, const double *z, const double *beta, double *p, hipStream_t s);
double l_packed_fro2(int n, const double *a, double *part, double *scal, hipStream_t s);
void l_zero(int64_t n, double *y, hipStream_t s);

// factor of the dense solve methods, kept until the matrix changes (as pede's mchdec decomposes
// only after a matrix pass and otherwise reuses the decomposition, src/pede.f90:8024-8047)
struct DenseFactor {
    int n = 0;
    int metsol = 0;      // method the factor was made for
    bool rev = false;    // factor of the index-reversed matrix (chdec2's pivot order)
    bool fp32 = false;   // FP32 factor (refinement in FP64); false: FP64 factor
    double rho = 0.0, anorm = 0.0;   // weight of the augmenting C^T C term, ||A + rho C^T C||_F bound
    int nrank = 0;
    double evmax = 0.0, evmin = 0.0;
    DBuf<double> a, w, work;
    DBuf<float> a32, w32, work32;
    DBuf<double> sc;     // FP32 factor: it factors D A D with D = diag(A)^-1/2 (unit diagonal)
    std::vector<double> piv;
    // v <- A^-1 v for nrhs columns of length n (leading dimension n) with the FP64 factor
    void solve64(double *v, int nrhs, hipStream_t s)
    {
        if (rev) l_reverse(n, v, nrhs, n, s);
        ldl_solve(n, a.p, n, w.p, work.p, v, nrhs, n, s);
        if (rev) l_reverse(n, v, nrhs, n, s);
    }
    // A^-1 = D (D A D)^-1 D
    void solve32(double *v, int nrhs, hipStream_t s)
    {
        l_scale_cols(n, sc.p, v, nrhs, n, s);
        if (rev) l_reverse(n, v, nrhs, n, s);
        ldl_solve32(n, a32.p, n, w32.p, work32.p, v, nrhs, n, s);
        if (rev) l_reverse(n, v, nrhs, n, s);
        l_scale_cols(n, sc.p, v, nrhs, n, s);
    }
};

// ---- index maps and matrix structure on the device (k_struct.hip) ----
// the compiled records on the device, as the structure kernels read them
struct StructIn {
    int64_t nrec = 0, neq = 0;
    const int64_t *rec_eq = nullptr, *rec_w = nullptr, *eq_sl = nullptr;   // rec_w: word range of each record
    const uint32_t *eq_n = nullptr;
    const int32_t *lab = nullptr;       // the record words as read (global words hold labels)
    const float *vf = nullptr;
    const double *vd = nullptr;
};
// labels in use: bitmap over [lmin, lmin + 32 nw) and the rank of every 32-bit word
struct LabelMap {
    int32_t lmin = 0;
    int64_t nw = 0;
    int64_t neq_glob = 0, nglob_words = 0;   // equations with global derivatives, global words
    DBuf<uint32_t> bits;
    DBuf<int64_t> wrank;
};
// group pairs in use: bitmap over the lower triangle (a, b <= a) at bit a (a + 1) / 2 + b
struct PairMap {
    int64_t nw = 0;
    DBuf<uint32_t> bits;
    DBuf<int64_t> wrank;
};
// group-block storage: blocks in row-major order of the lower block triangle
struct BlockDev {
    int64_t nblock = 0, nstored = 0, ncc = 0;
    DBuf<int64_t> brow, boff, ccol_ptr, cc_off;
    DBuf<int32_t> brg, bcol, bcf, cc_fn, cc_blk;
};
// parts of the block rows for the block product (groups <= 8; whole: one part a row): returns the
// entries of part
int64_t st_row_parts(int32_t ngroup, int64_t nblock, const int64_t *brow, const int32_t *bcol, const int64_t *boff, bool whole,
                     DBuf<RowPart> &part, DBuf<int64_t> &ptr, hipStream_t s);
// equation tables of the records (decodeNextMeasurement): fills in.neq, in.rec_eq, in.eq_sl,
// in.eq_n; error 20 names the first record that breaks the format
int64_t st_decode(StructIn &in, DBuf<int64_t> &rec_eq, DBuf<int64_t> &eq_sl, DBuf<uint32_t> &eq_n, hipStream_t s);
// labels -> total indices; c.labels (sorted) on the host; extra: labels of steering parameters,
// constraints and external measurements
void st_label_table(const StructIn &in, const std::vector<int32_t> &extra, LabelMap &map, std::vector<int32_t> &labels,
                    hipStream_t s);
// per record: sorted distinct total indices (gl lists), the position of every global word in its
// record's list (widx), the entry counters and the group-boundary flags (per record or per
// equation counting)
void st_record_lists(const StructIn &in, const LabelMap &map, int32_t ntot, bool per_record, DBuf<int32_t> &widx,
                     DBuf<int64_t> &rec_gl, DBuf<int32_t> &gl_tix, std::vector<int32_t> &ngl_rec,
                     std::vector<int64_t> &counters, std::vector<uint8_t> &bnd, hipStream_t s);
// per record: st[k * nrec + r], k = variables, segments, largest local index, local x global
// words, equations per variable, first group; cnt_r: values of its matrix update; sparse: the
// group pairs it couples into pm
// a context on a stream the caller keeps (serving workers reuse one stream per worker), or on
// a stream of its own when stream is null
int create_context(const mpgpu_options *opt, int32_t device, hipStream_t stream, mpgpu_ctx **out);
DevCache &context_memory(mpgpu_ctx *c);
// device bytes of a packed matrix of n rows and what a solve allocates beside it: the inversion a
// copy and a square matrix (1 + 2 packed), the FP64 factor a full matrix (2), the FP32 factor a full
// FP32 one (1) and, when the refinement does not converge, the FP64 factor as well; workspaces
inline int64_t full_storage_bytes(int metsol, int64_t n)
{
    int64_t mult = 2;
    switch (metsol) {
    case MPGPU_INVERSION: mult = n > 128 ? 4 : 2; break;
    case MPGPU_DECOMPOSITION: case MPGPU_LAPACK_PACKED: case MPGPU_LAPACK_UNPACKED: mult = 3; break;
    case MPGPU_CHOLESKY_FP32_IR: mult = 4; break;
    default: break;
    }
    return mult * (8 * n * (n + 1) / 2) + 4096 * n;
}
// FP32 values widened to FP64 (device to device)
void st_widen(const float *src, double *dst, int64_t n, hipStream_t s);
// residual monitoring: label of the first global word (0: none) and error of every equation
void st_eq_first(const StructIn &in, std::vector<int32_t> &lab, std::vector<double> &err, hipStream_t s);
// iterated entries cut: recount the global words of the equations without a low parameter
void st_entries_recount(const StructIn &in, const LabelMap &map, const std::vector<uint8_t> &low,
                        std::vector<int64_t> &counts, hipStream_t s);
void st_record_stats(const StructIn &in, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl,
                     const DBuf<int32_t> &gl_tix, const int32_t *var, const int32_t *group_of, int32_t ngroup,
                     int32_t max_ngl, bool sparse, PairMap &pm, std::vector<int32_t> &st, std::vector<int64_t> &cnt_r,
                     DBuf<int32_t> &d_st, hipStream_t s);
// storage: with the blocks' offsets and column lists
void st_blocks(PairMap &pm, int32_t ngroup, const int32_t *gfirst, const std::vector<int64_t> &extra_pairs, BlockDev &B,
               bool storage, hipStream_t s);
void st_pair_blocks(const StructIn &in, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix, const int32_t *var,
                    const int32_t *group_of, int32_t max_nseg, const DBuf<int32_t> &d_st, const PairMap &pm,
                    DBuf<int64_t> &rec_pb, DBuf<int32_t> &pair_blk, hipStream_t s);
// processing order: records stably sorted by their first parameter group
void st_order(int64_t nrec, int32_t ngroup, const DBuf<int32_t> &d_st, DBuf<int64_t> &order, std::vector<int64_t> &h_order,
              hipStream_t s);
// incidence lists of the batch order[q0, q1): ptr[nblock + 1], src[nsrc]
void st_incidence(const StructIn &in, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix, const int32_t *var,
                  const int32_t *group_of, int32_t max_nseg, const DBuf<int64_t> &order, const DBuf<int64_t> &rec_pb,
                  const DBuf<int32_t> &pair_blk, const DBuf<int64_t> &rec_cb, int64_t q0, int64_t q1, int64_t nblock,
                  int64_t *ptr, int64_t *src, int64_t nsrc, hipStream_t s);

// ---- records in row form (k_rows.hip) ----
struct RowStruct {
    // ncls: off-diagonal blocks whose lists are long, medium, short (k_rows_gather)
    struct Batch { int64_t q0, q1, unit0, nunit, inc0, npair, ncls[3]; };
    int64_t nq = 0, nrow = 0, nseg = 0, nunit = 0, npair = 0;
    int kp = 4, gp = 6, max_eq = 0;   // local and group columns of a row, most equations of a record
    bool dbl = false;
    DBuf<int32_t> n;                  // per record counts (k_rows_class)
    DBuf<int64_t> order, c;           // processing order; running sums of the counts in that order
    DBuf<RowHdr> hdr;
    DBuf<uint8_t> rows;
    DBuf<int32_t> eq_t0, ptix;
    DBuf<uint16_t> eq_pos, seq;
    DBuf<int4> seg;
    std::vector<Batch> batches;       // matrix build: batches of records and their incidence lists
    DBuf<uint32_t> ptr, perm;         // perm: order of the blocks in the gather
    DBuf<uint2> src;
    // units and side array of the largest batch: contents live only within a pass, so that an
    // allocation that fails between passes can have their memory (alloc_units)
    DBuf<uint8_t> unit;
    DBuf<double> side;
    size_t unit_bytes = 0, side_len = 0;
    bool in_pass = false;
    int64_t nblock = 0;               // full storage: the pairs of groups that some record couples
    DBuf<int64_t> brow;
    DBuf<int32_t> brg, bcol;
    void alloc_units()
    {
        unit.alloc(unit_bytes);
        side.alloc(side_len);
    }
    void free_units()
    {
        unit.release(); side.release();
    }
    void drop()
    {
        nq = 0;
        order.release(); c.release(); n.release(); hdr.release(); rows.release(); eq_t0.release(); ptix.release();
        eq_pos.release(); seq.release(); seg.release(); ptr.release(); perm.release(); src.release(); brow.release();
        brg.release(); bcol.release();
        free_units();
        batches.clear();
    }
    // device bytes of the incidence lists and the block order for nb blocks, with what their sorts need
    int64_t list_bytes(int64_t nb) const { return 8 * npair + 24 * std::min<int64_t>(npair, (int64_t)1 << 30) + 48 * nb; }
};
void rows_classify(const StructIn &in, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix,
                   const int32_t *band, const RowGroups &Q, RowStruct &S, std::vector<uint8_t> &cls, hipStream_t s);
void rows_build(const StructIn &in, const DBuf<int32_t> &widx, const DBuf<int64_t> &rec_gl, const DBuf<int32_t> &gl_tix,
                const RowGroups &Q, const std::vector<int64_t> &order, RowStruct &S, hipStream_t s);
void rows_incidence(RowStruct &S, const int32_t *group_of, const PairMap &pm, int64_t nblock, const int32_t *brg,
                    const int32_t *bcol, int64_t budget, const std::vector<int64_t> &upd, hipStream_t s);
hipError_t launch_rows(const RowStruct &S, const RowDev &R, const DevModel &M, const PassOpts &o, const RecOut &out, bool build,
                       int64_t q0, int64_t q1, hipStream_t s);
hipError_t launch_rows_gather(const RowStruct &S, size_t batch, int32_t ngroup, int64_t nblock, const int64_t *brow,
                              const int64_t *boff, const int32_t *brg, const int32_t *bcol, const int32_t *gfirst, double *mat,
                              double *vec, unsigned long long *cnt, hipStream_t s);

// ---- constraint elimination (mpgpu_qldec.cpp, k_qlelim.hip) ----
// device view of the reflectors: rows over parameter ranges, the transpose per parameter, the WY
// factor T and two m-vectors of scratch
struct QlDev {
    int32_t n = 0, m = 0;
    const int64_t *rf_ptr = nullptr, *tr_ptr = nullptr;
    const int32_t *rf_lo = nullptr, *rf_kn = nullptr, *tr_k = nullptr;
    const double *rf_val = nullptr, *rf_vk = nullptr, *tr_v = nullptr, *T = nullptr;
    double *w = nullptr, *u = nullptr;
};
struct QlElim {
    int32_t nvar = 0, ncon = 0, nfit = 0, nblk = 0;
    double evmin = 0.0, evmax = 0.0;
    std::vector<int> order;            // input constraint of each QL column (pede's sorted order)
    std::vector<int32_t> rcon, bcon;   // matConsRanges (4 per constraint), matConsBlocks (3 per block + end)
    std::vector<int64_t> ioffRow;
    std::vector<int32_t> ioffPar, irng;
    std::vector<double> matV, vecVk, matL;
    std::vector<int64_t> rf_ptr, tr_ptr;
    std::vector<int32_t> rf_lo, rf_kn, tr_k;
    std::vector<double> rf_val, rf_vk, tr_v, T;
    std::vector<double> vtvp;          // V^T V with entries of magnitude <= 16 eps cleared, unit diagonal
    DBuf<int64_t> d_rf_ptr, d_tr_ptr;
    DBuf<int32_t> d_rf_lo, d_rf_kn, d_tr_k;
    DBuf<double> d_rf_val, d_rf_vk, d_tr_v, d_T, d_w, d_u;
    QlDev dev;

    void build(int32_t nvar, const std::vector<std::vector<std::pair<int32_t, double>>> &con_tot,
               const std::vector<int32_t> &var_index);
    void upload(hipStream_t s);
    std::vector<double> bsub(const std::vector<double> &d) const;
    // coefficients of pede's band transform from X = V^T A V (column-major): Cf (row-major m x m)
    // and the diagonal weights D
    void band_coef(const std::vector<double> &X, std::vector<double> &Cf, std::vector<double> &D) const;

  private:
    void decompose();
    void wy();
};
void l_ql_apply(const QlDev &q, int trans, double *x, hipStream_t s);   // x <- Q x (0) or Q^T x (1)
bool ql_few(const QlDev &q);                 // few enough constraints for l_ql_op
void l_ql_op(const QlDev &q, int trans, int32_t nx, const double *x, double *y, int32_t ny, hipStream_t s);
void l_ql_pad(int32_t nfit, int32_t n, const double *x, double *e, hipStream_t s);
void l_ql_vtx_cols(const QlDev &q, const double *x, int64_t ldx, int32_t ncols, double *w, int64_t ldw, hipStream_t s);
void l_ql_vdense(const QlDev &q, double *Vd, hipStream_t s);
void l_ql_y(const QlDev &q, const double *Cf, double *P, hipStream_t s);
void l_ql_band(const QlDev &q, int32_t nfit, int32_t mb, const int32_t *india, const double *P, const double *S,
               double *band, hipStream_t s);

} // namespace mpgpu
