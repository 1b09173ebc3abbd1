/*
 * host_stub.c -- the kernel-level C-ABI (ptt_hip.h) on host memory without
 * arithmetic, to run the C host layer on a CPU and see which products it queues
 * where and what it allocates.  Factorisations report what the test sets
 * (stub_kappa, stub_deficient); spectra are flat.  Nothing here checks values.
 */
#include <stdlib.h>
#include <string.h>

#include "paratt.h"
#include "pattac.h"
#include "ptt_hip.h"

double stub_kappa = 1.5;
int stub_deficient = 0;
long stub_bad_chol = -1; /* the factorisation (from 0) that reports a condition of 1e7 */
long stub_side_inplace; /* in-place products queued on the side stream (Q = A T) */
long stub_main_inplace; /* the same on the main stream, c x c from the right */
long stub_chol, stub_tree_factors, stub_eigen, stub_mallocs;
long stub_frees; /* calls that free (each waits for the device) */
size_t stub_live, stub_peak;

static int on_side;

void stub_reset(void) {
    stub_side_inplace = stub_main_inplace = 0;
    stub_chol = stub_tree_factors = stub_eigen = stub_mallocs = stub_frees = 0;
    stub_peak = stub_live;
}

/* ---- memory: sizes in front of the block ---- */
void *ptt_hip_malloc(size_t bytes) {
    size_t *p = (size_t *)calloc(1, bytes + 64);
    if (!p) abort();
    p[0] = bytes;
    stub_mallocs++;
    stub_live += bytes;
    if (stub_live > stub_peak) stub_peak = stub_live;
    return p + 8;
}
void ptt_hip_free(void *p) {
    if (!p) return;
    size_t *q = (size_t *)p - 8;
    stub_live -= q[0];
    free(q);
}
void ptt_hip_free_many(int count, void *const *p) {
    for (int i = 0; i < count; i++) ptt_hip_free(p[i]);
    if (count > 0) stub_frees++;
}
static struct {
    void *p;
    size_t cap;
} slots[PTT_WS_NSLOTS];
void *ptt_hip_scratch(int slot, size_t bytes) {
    if (bytes > slots[slot].cap) {
        ptt_hip_free(slots[slot].p);
        slots[slot].p = ptt_hip_malloc(bytes);
        slots[slot].cap = bytes;
    }
    return slots[slot].p;
}
void ptt_hip_swap_tmp(int slot, double **buf, size_t *cap) {
    void *p = slots[slot].p;
    size_t c = slots[slot].cap;
    slots[slot].p = *buf;
    slots[slot].cap = *cap;
    *buf = (double *)p;
    *cap = c;
}
void ptt_hip_h2d(void *d, const void *s, size_t n) { memcpy(d, s, n); }
void ptt_hip_h2d_queued(void *d, const void *s, size_t n) { memcpy(d, s, n); }
void ptt_hip_d2h(void *d, const void *s, size_t n) { memcpy(d, s, n); }
void ptt_hip_d2d(void *d, const void *s, size_t n) { (void)d; (void)s; (void)n; }
void ptt_hip_copy(void *d, const void *s, size_t n) { memmove(d, s, n); }
static const void *d2h_src;
unsigned long long ptt_hip_d2h_begin(const void *s, size_t n) { (void)n; d2h_src = s; return 1; }
void ptt_hip_d2h_end(unsigned long long t, void *d, size_t n) { (void)t; memcpy(d, d2h_src, n); }
void ptt_hip_zero(void *p, size_t n) { memset(p, 0, n); }
void ptt_hip_sync(void) {}

/* ---- streams ---- */
int ptt_hip_side_enabled(void) { return 1; }
void ptt_hip_side_begin(void) { on_side = 1; }
void ptt_hip_side_end(int slot) { (void)slot; on_side = 0; }
void ptt_hip_side_wait(int slot) { (void)slot; }
void ptt_hip_side_join(void) {}

/* ---- products and factorisations ---- */
void ptt_hip_dgemm(char ta, char tb, int M, int N, int K, double alpha, const double *A, long lda,
                   const double *B, long ldb, double beta, double *C, long ldc) {
    (void)alpha; (void)B; (void)ldb; (void)beta; (void)lda; (void)ldc;
    if (ta == 'N' && tb == 'N' && A == C && M >= N && N == K) {
        if (on_side) stub_side_inplace++;
        else stub_main_inplace++;
    }
}
void ptt_hip_trmm_small(int c, const double *A, const double *B, double *C) {
    (void)c; (void)A; (void)B; (void)C;
}
void ptt_hip_gram(char t, int c, long n, const double *A, long lda, double *G) {
    (void)t; (void)c; (void)n; (void)A; (void)lda; (void)G;
}
void ptt_hip_gram32(char t, int c, long n, const double *A, long lda, double *G) {
    ptt_hip_gram(t, c, n, A, lda, G);
}
void ptt_hip_chol_qr_factor(int c, const double *G, double shift, double tiny, double *R, double *T,
                            int *info, double *dinfo, int want) {
    (void)c; (void)G; (void)shift; (void)tiny; (void)R; (void)T; (void)want;
    const int bad = stub_chol++ == stub_bad_chol;
    info[0] = stub_deficient;
    dinfo[0] = 0.0;
    dinfo[1] = bad ? 1e7 : stub_kappa;
    dinfo[2] = stub_deficient;
    dinfo[3] = 1.0;
}
static void flat(int k, int cap, double *sig, int *iout) {
    for (int j = 0; j < k; j++) sig[j] = 1.0;
    iout[0] = k;
    iout[1] = cap < 1 ? 1 : cap < k ? cap : k;
    iout[2] = 1;
}
void ptt_hip_syev_gram(int c, const double *G, double *sig, double *U, long ldu, int *ci, int *iout,
                       double *dinfo, double delta, int cap, double budget) {
    (void)G; (void)U; (void)ldu; (void)ci; (void)delta; (void)budget;
    stub_eigen++;
    flat(c, cap, sig, iout);
    dinfo[5] = 0.0;
    dinfo[6] = 1.0;
    dinfo[7] = c;
}
void ptt_hip_svd_jacobi(int m, int k, double *A, long lda, double *sig, double *U, long ldu,
                        double *V, long ldv, double ls, double delta, int cap, int *iout) {
    (void)m; (void)A; (void)lda; (void)U; (void)ldu; (void)V; (void)ldv; (void)ls; (void)delta;
    flat(k, cap, sig, iout);
}
void ptt_hip_svd_right(int k, const double *R, long ldr, double *X, double *sig, double *V,
                       long ldv, double delta, int cap, int *iout) {
    (void)R; (void)ldr; (void)X; (void)V; (void)ldv; (void)delta;
    flat(k, cap, sig, iout);
}
void ptt_hip_svd_right_from(int k, const double *R, long ldr, const double *U, long ldu, double *X,
                            double *sig, double *V, long ldv, double delta, int cap, int *iout) {
    (void)U; (void)ldu;
    ptt_hip_svd_right(k, R, ldr, X, sig, V, ldv, delta, cap, iout);
}
void ptt_hip_svd_factors(int m, int r, const int *dr, const double *U, long ldu, const double *sig,
                         double ws, double *W, double *US) {
    (void)m; (void)r; (void)dr; (void)U; (void)ldu; (void)sig; (void)ws; (void)W; (void)US;
}
void ptt_hip_svd_factors_perm(int m, int r, const int *ci, const double *U, long ldu,
                              const double *sig, double ws, double *W, double *US) {
    ptt_hip_svd_factors(m, r, ci, U, ldu, sig, ws, W, US);
}
void ptt_hip_sumsq(int m, int n, const double *A, long lda, double *out) {
    (void)m; (void)n; (void)A; (void)lda;
    *out = 1.0;
}
double ptt_hip_maxabs(const double *A, long n) { (void)A; (void)n; return 1.0; }
int ptt_hip_tsqr_plan(int c, long rows, ptt_tsqr_plan *pl) {
    memset(pl, 0, sizeof *pl);
    pl->c = c;
    pl->rows = rows;
    pl->levels = 1;
    pl->fsize = 1024;
    return 0;
}
void ptt_hip_tsqr_factor(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                         long rpr, double *F, double *S, double *R, int *e) {
    (void)pl; (void)A; (void)rs; (void)cs; (void)drho; (void)rpr; (void)F; (void)S; (void)e;
    if (R) stub_tree_factors++;
}
void ptt_hip_tsqr_svd(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                      long rpr, double *F, double *S, double delta, int cap, double *sig, int *info,
                      int *rho, double *X, double *US, double *W, double *Y, double alpha) {
    (void)A; (void)rs; (void)cs; (void)drho; (void)rpr; (void)F; (void)S; (void)delta; (void)X;
    (void)US; (void)W; (void)Y; (void)alpha;
    flat(pl->c, cap, sig, info);
    *rho = info[1];
}
void ptt_hip_tsqr_finish(const ptt_tsqr_plan *p0, const double *A0, const int *d0, long r0,
                         const double *F0, const double *S0, const int *rho0, double *W0,
                         double *Y0, double al0, const ptt_tsqr_plan *p1, const double *A1,
                         const double *F1, const double *S1, const double *US1, const int *q1,
                         double *W1, double *Y1, double al1) {
    (void)p0; (void)A0; (void)d0; (void)r0; (void)F0; (void)S0; (void)rho0; (void)W0; (void)Y0;
    (void)al0; (void)p1; (void)A1; (void)F1; (void)S1; (void)US1; (void)q1; (void)W1; (void)Y1;
    (void)al1;
}

/* ---- streaming: nothing to do ---- */
void ptt_hip_scale(double *p, long n, double a) { (void)p; (void)n; (void)a; }
void ptt_hip_set_diag(double *A, int m, long lda, double a) { (void)A; (void)m; (void)lda; (void)a; }
void ptt_hip_transpose(int m, int n, const double *A, long lda, double *B, long ldb, double a) {
    (void)m; (void)n; (void)A; (void)lda; (void)B; (void)ldb; (void)a;
}
void ptt_hip_copy2d(int m, int n, const double *A, long lda, double *B, long ldb, double a) {
    ptt_hip_transpose(m, n, A, lda, B, ldb, a);
}
void ptt_hip_copy_train(int d, double *const *dst, double *const *src, const long *count) {
    (void)d; (void)dst; (void)src; (void)count;
}
void ptt_hip_gauss_fill(double *d, long n, uint64_t seed, int core, double s) {
    (void)d; (void)n; (void)seed; (void)core; (void)s;
}
void ptt_hip_sym_sort_perm(int c, const double *G, double *Gp, int *perm) {
    (void)c; (void)G; (void)Gp; (void)perm;
}
void ptt_hip_permute_rows(int m, int n, const int *p, const double *s, long ls, double *d, long ld) {
    (void)m; (void)n; (void)p; (void)s; (void)ls; (void)d; (void)ld;
}
void ptt_hip_unpermute_rows(int m, int n, const int *p, const double *s, long ls, double *d, long ld) {
    (void)m; (void)n; (void)p; (void)s; (void)ls; (void)d; (void)ld;
}
void ptt_hip_drop_small_cols(int m, int k, double *L, long ld, double b, double *dropped) {
    (void)m; (void)k; (void)L; (void)ld; (void)b;
    *dropped = 0.0;
}

/* not reached: the formal sums are not among the sources compiled */
void attacFormalSum(const int d, const int *n, const int *rx, double *const *x, const int *ry,
                    double *const *y, int *rz, double **z) {
    (void)d; (void)n; (void)rx; (void)x; (void)ry; (void)y; (void)rz; (void)z;
    abort();
}
