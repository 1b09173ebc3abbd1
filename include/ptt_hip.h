/*
 * ptt_hip.h -- the thin C-ABI between the C host layer (paratt.h API) and
 * the hand-written gfx950 HIP kernels.  Plain pointers and sizes only.
 *
 * All kernel launchers are asynchronous on the library's single HIP stream
 * (created at default priority on first use); ptt_hip_sync() waits for it.
 * Column-major everywhere; "ld" is the leading dimension in elements.
 * Any HIP runtime error is fatal: it is printed to stderr and the process
 * exits with status 1 (the reference's error convention, paratt.c:1642-1645).
 */
#ifndef PARATT_AMD_PTT_HIP_H
#define PARATT_AMD_PTT_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- runtime ---- */
void ptt_hip_init(void);
int ptt_hip_initialized(void);      /* 1 after ptt_hip_init */
void ptt_hip_noalloc_setup(void);   /* part of ptt_hip_init: fixed workspace address */
/* Device memory; freed blocks are kept for reuse (bounded, see runtime.hip)
 * and given back to the device by ptt_hip_trim.  Freeing waits for all device
 * work, once per call. */
void *ptt_hip_malloc(size_t bytes);
void ptt_hip_free(void *p);
void ptt_hip_free_many(int count, void *const *p);
void ptt_hip_trim(void);
void ptt_hip_h2d(void *dst, const void *src, size_t bytes);       /* blocking */
/* The same, stream-ordered: src is read before the call returns, dst is
 * written in order with the main stream's work (up to 64 KiB; blocking above). */
void ptt_hip_h2d_queued(void *dst, const void *src, size_t bytes);
void ptt_hip_d2h(void *dst, const void *src, size_t bytes);       /* blocking */
void ptt_hip_d2d(void *dst, const void *src, size_t bytes);       /* async */
/* A device-to-host read of at most 64 KiB in two halves: begin queues the
 * copy on the main stream and returns a ticket; end waits for that copy only
 * (kernels queued after begin keep running) and copies the bytes to dst.
 * One read may be open at a time; no ptt_hip_d2h in between. */
unsigned long long ptt_hip_d2h_begin(const void *src, size_t bytes);
void ptt_hip_d2h_end(unsigned long long ticket, void *dst, size_t bytes);
void ptt_hip_zero(void *p, size_t bytes);                         /* async fill kernel */
/* Blocking copy between any two host or device addresses. */
void ptt_hip_copy(void *dst, const void *src, size_t bytes);
/* 1 when the library runs in host-visible mode (environment variable
 * PARATT_AMD_HOST_VISIBLE=1 at first use): every allocation above is then
 * pinned host memory that the GPU accesses through the same address, so
 * host code may read and write cores directly between calls. */
int ptt_hip_host_visible(void);
void ptt_hip_sync(void);  /* waits for the main and the side stream */
/* A second stream for work off the critical path.  side_begin orders the side
 * stream after everything queued so far on the main stream and sends later
 * launches to it; side_end(slot) records the side stream's progress in event
 * `slot` (0 or 1) and returns launches to the main stream; side_wait(slot)
 * makes the main stream wait for that event; side_join makes the main stream
 * wait for all side work.  Only kernel launches (no copies) belong between
 * side_begin and side_end.  side_enabled is 0 when the environment sets
 * PARATT_AMD_NO_SIDE_STREAM=1. */
int ptt_hip_side_enabled(void);
void ptt_hip_side_enable(int on); /* switch the side stream on or off (waits first) */
void ptt_hip_side_begin(void);
void ptt_hip_side_end(int slot);
void ptt_hip_side_wait(int slot);
void ptt_hip_side_join(void);
/* Grow-only device scratch slots owned by the library.  The returned pointer
 * is valid until the next call for the same slot with a larger size. */
enum { PTT_WS_GRAM = 0, PTT_WS_SMALL, PTT_WS_TMP, PTT_WS_TMP2, PTT_WS_INT,
       PTT_WS_COEF, PTT_WS_SKETCH, PTT_WS_SMALL2, PTT_WS_RSK, PTT_WS_SIDE, PTT_WS_EIG,
       PTT_WS_RES, PTT_WS_RSIDE, PTT_WS_ROUT0, PTT_WS_ROUT1, PTT_WS_TREE, PTT_WS_QFACT,
       PTT_WS_NSLOTS };
void *ptt_hip_scratch(int slot, size_t bytes);
/* Exchange the buffer of the TMP slot with a caller buffer: on return *buf
 * points at the old scratch (capacity *cap_bytes updated) and the slot owns
 * the caller's old buffer.  Used to make out-of-place results in place. */
void ptt_hip_swap_tmp(int slot, double **buf, size_t *cap_bytes);
size_t ptt_hip_scratch_cap(int slot);

/* ---- profiling: HIP events around launches, per kernel name ---- */
void ptt_hip_prof_enable(int on);
void ptt_hip_prof_reset(void);
/* Record only launches named `name` (NULL or "" records every launch): keeps
 * the event overhead out of a timed region while one kernel is measured. */
void ptt_hip_prof_only(const char *name);
/* Returns 1 and fills count / total_ms if `name` was recorded (syncs). */
int ptt_hip_prof_get(const char *name, int *count, double *total_ms);
/* Algorithmic flops and bytes credited to `name` (syncs). */
int ptt_hip_prof_get_work(const char *name, double *flops, double *bytes);
/* Names recorded so far, '\n'-separated, into buf (truncated to len). */
void ptt_hip_prof_names(char *buf, int len);
/* Wall-clock of the stream between two markers, in ms (syncs). */
void ptt_hip_timer_start(void);
double ptt_hip_timer_stop(void);

/* ---- streaming kernels (HBM-bound) ---- */
/* Seeded N(0,1)*scale fill of `count` entries, element e of core `core`
 * of the TT with seed `seed` (same stream as the CPU generator). */
void ptt_hip_gauss_fill(double *dst, long count, uint64_t seed, int core,
                        double scale);
void ptt_hip_scale(double *p, long count, double alpha);
/* Block placement of one core of z = a*x (+) b*y.
 * kind 0: first core (column concat, scaled by a / b); kind 1: interior
 * (block diagonal); kind 2: last core (row concat). */
void ptt_hip_axpby_core(int kind, int n, int rx0, int rx1, const double *x,
                        int ry0, int ry1, const double *y, double a, double b,
                        double *z);
/* The same for d cores in as few launches as their count allows: core k has
 * kind[k], modes n[k] and ranks rx[k], rx[k+1] / ry[k], ry[k+1]. */
void ptt_hip_axpby_train(int d, const int *kind, const int *n, const int *rx,
                         double *const *x, const int *ry, double *const *y, double a,
                         double b, double *const *z);
/* dst[k][0..count[k]) = src[k][0..count[k]) for d cores. */
void ptt_hip_copy_train(int d, double *const *dst, double *const *src, const long *count);
/* S = sum_i D_i u as a rank-2r train of d cores: first [D u | u], interior
 * [[u, 0], [D u, u]], last [u; D u] (d = 1: D u), D the periodic 3-point
 * stencil of kind 0 below (host coefficients). */
void ptt_hip_mode_sum_train(int d, const int *n, const int *r, double *const *u,
                            const double *sten3, double *const *s);
/* Kronecker of every mode slice: z[(ry0*ax+ay), j, (ry1*bx+by)]. */
void ptt_hip_hadamard_core(int n, int rx0, int rx1, const double *x, int ry0,
                           int ry1, const double *y, double *z);
/* f[a,j,b] *= v[j]  (v on device). */
void ptt_hip_diag_core(int r0, int n, int r1, const double *v, double *f);
/* Mode stencils, out-of-place: g = op(f).  coef on device.
 * kind 0: pattac periodic (reference ghost-counter semantics),
 * kind 1: attac periodic (exact wrap), kind 2: cdf (mirror ghosts). */
void ptt_hip_stencil_core(int kind, int r0, int n, int r1, const double *sten,
                          int slen, const double *f, double *g);
/* Lax-Friedrichs-type flux (coef = [c(n), gc(2), s(n)]) and Lax-Wendroff
 * RHS (coef = [c(n), gc(2), bw(n+1), s(n)]). */
void ptt_hip_lf_flux_core(int r0, int n, int r1, const double *coef, double dt,
                          double dx, const double *f, double *g);
void ptt_hip_lw_rhs_core(int r0, int n, int r1, const double *coef, double dt,
                         double dx, const double *f, double *g);
/* Copy an m x n block with strides, optional scaling: B = alpha * A. */
void ptt_hip_copy2d(int m, int n, const double *A, long lda, double *B, long ldb,
                    double alpha);
/* B (n x m) = alpha * A^T (A m x n). */
void ptt_hip_transpose(int m, int n, const double *A, long lda, double *B,
                       long ldb, double alpha);
/* p[0..count) = v. */
void ptt_hip_fill(double *p, long count, double v);
/* A[i + i*lda] = alpha for i < m (other entries untouched). */
void ptt_hip_set_diag(double *A, int m, long lda, double alpha);
/* Squared Frobenius norm of an m x n block, result to device *out. */
void ptt_hip_sumsq(int m, int n, const double *A, long lda, double *out);

/* ---- dense linear algebra (FP64, MFMA) ---- */
/* C = alpha*op(A)*op(B) + beta*C.  ta/tb: 'N' or 'T'.  C may alias A (when
 * N fits one column tile) or B (when M fits one row tile): see gemm.hip. */
void ptt_hip_dgemm(char ta, char tb, int M, int N, int K, double alpha,
                   const double *A, long lda, const double *B, long ldb,
                   double beta, double *C, long ldc);
/* One mode of an inner product: out (rx1 x ry1) = s sum_j X_j^T a Y_j over the n
 * mode indices of the cores x (rx0 x n x rx1) and y (ry0 x n x ry1), a rx0 x ry0.
 * out may be a.  Returns 0, having done nothing, beyond ranks of 64. */
int ptt_hip_dot_mode(int n, int rx0, int rx1, int ry0, int ry1, const double *a, const double *x,
                     const double *y, double s, double *out);
/* Gram matrices with a split over the long dimension:
 * trans 'T': G (c x c) = A^T A for A (m x c, lda);
 * trans 'N': G (c x c) = A A^T for A (c x w, lda). */
void ptt_hip_gram(char trans, int c, long len, const double *A, long lda,
                  double *G);
/* The same for c <= 128 by the symmetric Gram kernel (upper 16 x 16 blocks
 * spread over the waves of each slab), FP64 throughout. */
void ptt_hip_gram_syrk(char trans, int c, long len, const double *A, long lda,
                       double *G);
/* Mixed precision: the Gram from FP32 inputs with FP32 accumulation inside
 * each slab (v_mfma_f32_16x16x4f32), slabs summed in FP64.  The input is
 * scaled by the power of two that brings its largest |entry| to [1, 2)
 * before rounding to FP32, and the result scaled back.  c <= 128; A must be
 * contiguous (lda = len for 'T', lda = c for 'N'). */
void ptt_hip_gram32(char trans, int c, long len, const double *A, long lda, double *G);

/* max |A_i| over count contiguous doubles, returned to the host (waits for
 * the library's queued work). */
double ptt_hip_maxabs(const double *A, long count);

/* Jacobi-scaled, guarded Cholesky of a c x c SPD Gram G (ld c):
 * D = sqrt(diag G); (D^-1 G D^-1 + shift*I) = Rs^T Rs; pivots below
 * `tiny` mark the index deficient (row of R and column of T set to 0).
 * Outputs (ld c): R = Rs*D (upper), T = D^-1 * Rs^-1 (upper, deficient
 * columns 0) so that A*T has orthonormal columns and A = (A*T)*R.
 * info[0] = dinfo[2] = number of deficient pivots, dinfo[0] =
 * ||Rs||_F*||Rs^-1||_F, dinfo[1] = 2-norm condition of Rs by power
 * iteration when want_kappa (else 0), dinfo[3] = max_j D_j^2 (the Gram's
 * largest diagonal entry).  T may be NULL when only R is needed: then no
 * inverse is formed and dinfo[0] = dinfo[1] = 0.  dinfo holds 4 doubles. */
void ptt_hip_chol_qr_factor(int c, const double *G, double shift, double tiny,
                            double *R, double *T, int *info, double *dinfo,
                            int want_kappa);

/* One-sided Jacobi SVD of A (m x k, lda, m >= k), FP64.
 * On return: sig[0..k) descending, U (m x k, ldu) left vectors,
 * V (k x k, ldv) right vectors if V != NULL.  Also the numerical rank
 * numrank (sig_j > sqrt(k)*eps*sig_0) and the truncation rank by the
 * reference's tail rule (pattac.c:468-481) applied to sig*exp(log_scale)
 * against delta, capped by min(k, cap), floor 1: written to iout[0]=numrank,
 * iout[1]=rho, iout[2]=sweeps; iout needs 5 ints.  Exactly-zero columns of
 * A are excluded from the rotations (their sigma is 0).  A is not changed.
 * Small k: one wave or one workgroup, columns in LDS; larger k: blocks of
 * columns over many workgroups, with one host read of a convergence flag per
 * sweep. */
void ptt_hip_svd_jacobi(int m, int k, double *A, long lda, double *sig,
                        double *U, long ldu, double *V, long ldv,
                        double log_scale, double delta, int cap, int *iout);
/* Singular values (k, descending) and right singular vectors (V, k x k, ldv;
 * columns of zero singular values are zero) of L = R^T, R upper triangular k x k
 * (ldr), k <= 128; X: k x k scratch.  Content below u times the largest column
 * is dropped.  iout = {numerical rank, tail-rule rank (against delta and cap),
 * sweeps} as in ptt_hip_svd_jacobi; iout needs 5 ints. */
void ptt_hip_svd_right(int k, const double *R, long ldr, double *X, double *sig, double *V,
                       long ldv, double delta, int cap, int *iout);
/* The same for k <= 192 from approximate left singular vectors U (k x k, ldu,
 * orthogonal, any order; may be V): nothing is dropped. */
void ptt_hip_svd_right_from(int k, const double *R, long ldr, const double *U, long ldu, double *X,
                            double *sig, double *V, long ldv, double delta, int cap, int *iout);
/* From U (m x k, ldu) and sig: W (rho x m, ld rho) = diag(1/sig) U_rho^T
 * scaled by wscale, and US (m x rho, ld m) = U_rho diag(sig).
 * rho is read from device *drho, or is rhomax when drho is NULL.  Either
 * output may be NULL. */
void ptt_hip_svd_factors(int m, int rhomax, const int *drho, const double *U,
                         long ldu, const double *sig, double wscale, double *W,
                         double *US);
/* Eigen-decomposition of a symmetric positive semi-definite c x c Gram G
 * (ld c, c <= 192): Householder tridiagonalisation, divide and conquer,
 * back transformation.  sig[q] = sqrt(lambda_q) in descending order; the
 * eigenvector of sig[q] is column colidx[q] (device ints) of U (c x c, ldu).
 * The smallest eigenvalues whose sum is at most budget * lambda_max are set
 * to zero (dinfo[5] = their sum); iout[0] = numerical rank (sig_q >
 * sqrt(c) eps sig_0), iout[1] = the reference's tail-rule rank against
 * delta, capped by min(c, cap), floor 1 (pattac.c:468-481), iout[2] = most
 * secular-equation iterations of one root; dinfo[6] = max |G_ij|,
 * dinfo[7] = trace(G).  With a NaN or an infinity in G's upper triangle every
 * sig is NaN and the numerical rank 0. */
void ptt_hip_syev_gram(int c, const double *G, double *sig, double *U, long ldu, int *colidx,
                       int *iout, double *dinfo, double delta, int cap, double budget);
/* ptt_hip_syev_gram without any allocation: same kernels, same results, the
 * workspace in a fixed device array of the library (one per GPU, about
 * 0.5 MB, held until the process ends).  No counterpart in the reference;
 * for callers that cannot allocate (code under HIP graph capture, serving
 * loops, harnesses that forbid hipMalloc).  The library must be set up
 * first (ptt_hip_init, which may allocate; returns -2 otherwise); c above 128
 * is rejected with a message (returns -1); 0 on success.  Calls that overlap
 * on one GPU share the array and race: serialise them (the library's stream
 * does, within one process). */
int ptt_hip_syev_gram_noalloc(int c, const double *G, double *sig, double *U, long ldu,
                              int *colidx, int *iout, double *dinfo, double delta, int cap,
                              double budget);
/* As ptt_hip_svd_factors for the first rho eigenpairs of ptt_hip_syev_gram:
 * W (rho x m, ld rho) = wscale diag(1/sig) U[:, colidx]^T, US (m x rho, ld m)
 * = U[:, colidx] diag(sig). */
void ptt_hip_svd_factors_perm(int m, int rho, const int *colidx, const double *U, long ldu,
                              const double *sig, double wscale, double *W, double *US);
/* ---- low-rank bonds: Householder trees (c <= 32 columns) ----------------------
 * The rows are cut into blocks, factored one workgroup each (level 0), their
 * c x c factors stacked and factored in turn up to a single block (the root).
 * F (pl->fsize doubles) and S (pl->ssize) belong to one factorisation and are
 * read by its applications. */
enum { PTT_TSQR_LEVELS = 6 };
typedef struct {
    int c, levels;
    long rows, fsize, ssize;
    int nblk[PTT_TSQR_LEVELS], brows[PTT_TSQR_LEVELS];
    long lrows[PTT_TSQR_LEVELS], foff[PTT_TSQR_LEVELS], soff[PTT_TSQR_LEVELS];
} ptt_tsqr_plan;
/* Returns 0, or -1 when the tree would be too deep. */
int ptt_hip_tsqr_plan(int c, long rows, ptt_tsqr_plan *pl);
/* A (element (row, col) at row * rs + col * cs) = Q R: the reflectors overwrite
 * A.  drho (may be NULL): the matrix has rows_per_rank * *drho rows, at most
 * pl->rows.  R (c x c, ld c) receives the factor, divided by 2^e where its
 * magnitude would leave FP64's safe range, e added to the device int *escale;
 * R NULL leaves the root to ptt_hip_tsqr_svd. */
void ptt_hip_tsqr_factor(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                         long rows_per_rank, double *F, double *S, double *R, int *escale);
/* The root of M^T = Q R (A = M, rs = c, cs = 1) and the SVD of L = R^T:
 * singular values (32, device), info = {numerical rank, rank kept by the tail
 * rule against delta and cap, sweeps, columns factored}, *rho = the rank kept,
 * X = the right singular vectors of L (c x rho, ld 32), US = U Sigma (row i at
 * i * 32), and the root's rows of Q X in W (2 * lrows[1] * 32 doubles).  A tree
 * of one level writes alpha (Q X)^T to Y (rho x rows) instead. */
void ptt_hip_tsqr_svd(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                      long rows_per_rank, double *F, double *S, double delta, int cap,
                      double *sig, int *info, int *rho, double *X, double *US, double *W,
                      double *Y, double alpha);
/* The rest of both applications of a right-to-left bond in as few launches as
 * their trees allow: Y0 (rho x rows) = alpha0 (Q0 X)^T below the root of pl0
 * (after ptt_hip_tsqr_svd; nothing for one level), and Y1 (rows x *p1,
 * column-major) = alpha1 Q1 US1 for the left-to-right tree pl1 (A1 column-major;
 * pl1 may be NULL; F1 NULL: A1 is an explicit Q and Y1 = alpha1 A1 US1).  W0,
 * W1: as W above, per tree. */
void ptt_hip_tsqr_finish(const ptt_tsqr_plan *pl0, const double *A0, const int *drho0,
                         long rows_per_rank0, const double *F0, const double *S0,
                         const int *rho0, double *W0, double *Y0, double alpha0,
                         const ptt_tsqr_plan *pl1, const double *A1, const double *F1,
                         const double *S1, const double *US1, const int *p1, double *W1,
                         double *Y1, double alpha1);
/* ---- rank-predictor network (FP32, 18 -> 64 -> 64 -> 64 -> 1, tanh-GELU) ----
 * X: nsamp x 18 row-major, Y: nsamp targets, P: ptt_hip_mlp_nparam() floats. */
int ptt_hip_mlp_nparam(void);
void ptt_hip_mlp_forward(int nsamp, const float *X, const float *P, float *out);
/* grad (nparam floats) and loss (1 float) are overwritten: mean-squared
 * error gradient over the batch. */
void ptt_hip_mlp_grad(int nsamp, const float *X, const float *Y, const float *P,
                      float *grad, float *loss);
void ptt_hip_mlp_adam(float *P, const float *grad, float *m, float *v, float lr,
                      int t);
/* Gp = G[perm, perm] for the c x c matrix G (ld c) with perm ordering the
 * diagonal descending (ties by index), perm (c ints, device) written too;
 * c <= 1024. */
void ptt_hip_sym_sort_perm(int c, const double *G, double *Gp, int *perm);
/* Zeroes the smallest-norm columns of L (m x k, ld; k <= 1024) whose squared
 * norms sum to at most budget * (largest squared column norm); the dropped
 * sum goes to device *dropped. */
void ptt_hip_drop_small_cols(int m, int k, double *L, long ld, double budget, double *dropped);
/* dst[perm[i] + j*ldd] = src[i + j*lds] for i < m, j < n. */
void ptt_hip_unpermute_rows(int m, int n, const int *perm, const double *src, long lds,
                            double *dst, long ldd);
/* dst[i + j*ldd] = src[perm[i] + j*lds] for i < m, j < n (gather). */
void ptt_hip_permute_rows(int m, int n, const int *perm, const double *src, long lds,
                          double *dst, long ldd);
/* Small c x c triangular product C = A*B (upper times upper), ld c. */
void ptt_hip_trmm_small(int c, const double *A, const double *B, double *C);

/* ---- quadrature along one mode, entry evaluation (FP64, bit-exact) ----
 * In place on the r0 x n x r1 core f, sequentially along every fiber
 * (a, :, b); w and scale are n-vectors on the device.
 * kind 0: weighted cumulative sum, g[j] = sum_{j'<=j} w[j'] f[j'];
 * kind 1: trapezoid rule, g[0] = 0, g[j] = g[j-1] + 0.5 w[j] (f[j-1] + f[j]);
 * kind 2: kind 1 plus f[j] * scale[j] (scale unused otherwise). */
void ptt_hip_mode_scan(int kind, int r0, int n, int r1, const double *w, const double *scale,
                       double *f);
/* C[i + ldc j + sC q] = sum_k A[i + lda k + sA q] * B[k + ldb j + sB q],
 * summed over k in order from 0.0 (i < M, j < N, q < batch). */
void ptt_hip_seq_gemm(int M, int N, int K, int batch, const double *A, long lda, long sA,
                      const double *B, long ldb, long sB, double *C, long ldc, long sC);
/* Entry (idx[0..d)) of the TT with device cores `cores`: chain of
 * matrix-vector products from the last core to the first.  vec: device
 * scratch of max rank doubles.  *out (host) receives the value (syncs). */
void ptt_hip_tt_entry(int d, const int *n, const int *r, double *const *cores, const int *idx,
                      double *vec, double *out);

#ifdef __cplusplus
}
#endif
#endif
