/*
 * round.c -- TT rounding on the GPU: left-to-right orthogonalisation and
 * right-to-left SVD truncation of device-resident cores.
 *
 * Follows pattacTruncate (pattac.c:590-675): the reference scales every core
 * by 1/sqrt(n_k), left-orthogonalises (pattac.c:244-294), truncates
 * right-to-left with tolerance abs_tol/sqrt(d-1) per bond (pattac.c:297-522)
 * and scales back by sqrt(n_k).  Here those scalings are folded into the
 * alpha of the GEMMs that produce each core, so every intermediate has the
 * reference's magnitude and no extra pass over the tensor is made.
 *
 * Factorizations (the MPI TSQR tree at one rank is a single dgeqrf/dgelqf,
 * tsqr.c:541-714, 1048-1222) are Cholesky-QR on the matrix cores:
 *   1 pass  when the Jacobi-scaled Gram is well conditioned (kappa <= 30):
 *           orthogonality error ~ u*kappa^2 <= 1e-13;
 *   2 passes (CholeskyQR2) when kappa <= 1e6;
 *   3 passes (shifted CholeskyQR3, Fukaya et al., SISC 2020) otherwise,
 *           which covers numerically rank-deficient cores.
 * The bond SVD is a one-sided Jacobi SVD of the r x r triangular factor;
 * in the well-conditioned case the new core is Sigma^-1 U^T times the old
 * core (one GEMM, no explicit Q), otherwise V^T times the explicit Q.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "paratt.h"
#include "paratt_amd.h"
#include "attac.h"
#include "ptt_hip.h"
#include "ptt_host.h"

#define KAPPA_ONE_PASS 30.0
/* Largest accepted estimate of the Gram route's subspace error (rtl_step_fast). */
#define FAST_EST_MAX 1.0e-13
/* Budget, in units of rows * u * (largest squared column norm), of the
 * factor columns the Gram route zeroes before its SVD. */
#define FAST_DROP 8.0
#define CHOLQR_MAX_PASSES 6
#define KAPPA_TWO_PASS 1.0e6
#define SKETCH_OVERSAMPLE 8

static paratt_amd_round_stats g_stats;

/* Leaf precision of the left-to-right Cholesky-QR: 0 FP64, 1 FP32 first
 * pass with an FP64 refinement. */
static int g_leaf32 = 0;

void paratt_amd_set_leaf_precision(int fp32_first_pass) { g_leaf32 = fp32_first_pass ? 1 : 0; }
int paratt_amd_leaf_precision(void) { return g_leaf32; }

void paratt_amd_last_round_stats(paratt_amd_round_stats *out) { *out = g_stats; }

/* Per-bond spectrum record of the last rounding (bond i = 1..d-1, i < 64):
 * [0..15] sigma_{rho-13+j} (0 outside the spectrum), [16] sigma_0,
 * [17] rho, [18] incoming rank, [19] 1 if the bond was set by a sketch. */
#define SPEC_W 20
static double g_spec[64][SPEC_W];

void paratt_amd_last_round_spectra(double *out) { memcpy(out, g_spec, sizeof g_spec); }

/* Every bond's whole spectrum is wanted (ptt_host_whole_spectra). */
static int g_whole_spectra = 0;
void ptt_host_whole_spectra(int on) { g_whole_spectra = on; }

/* The leading singular values of the current bond as the step brought them
 * to the host for its decisions (g_hsig_n = 0: not brought), reused by the
 * statistics and the spectrum record instead of another round trip. */
static double g_hsig[128];
static int g_hsig_n = 0;
static void keep_hsig(const double *sig, int n) {
    g_hsig_n = n < 128 ? n : 128;
    memcpy(g_hsig, sig, sizeof(double) * (size_t)g_hsig_n);
}

/* Sketched right-to-left steps: per-bond predicted ranks (NULL: none) and
 * counters {attempted, accepted} of the last rounding. */
static const int *g_pred = NULL;
static int g_sketch_counts[2];
static uint64_t g_sketch_seed = 0x5eed0001ULL;

void paratt_amd_last_sketch_counts(int *out) {
    out[0] = g_sketch_counts[0];
    out[1] = g_sketch_counts[1];
}

/* Small device workspace for one step: matrices up to c x c. */
typedef struct {
    double *G, *R1, *T1, *R2, *T2, *R3, *T3, *Racc, *Rtmp, *L, *U, *V, *sig, *W, *US, *dinfo;
    int *iinfo; /* [0] deficiency, [1..3] svd out */
    int cap;
} step_ws;

static step_ws get_ws_slot(int c, int slot) {
    step_ws w;
    size_t cc = (size_t)c * c;
    double *base = (double *)ptt_hip_scratch(slot, sizeof(double) * (15 * cc + 2 * (size_t)c + 128));
    w.G = base;
    w.R1 = w.G + cc;
    w.T1 = w.R1 + cc;
    w.R2 = w.T1 + cc;
    w.T2 = w.R2 + cc;
    w.R3 = w.T2 + cc;
    w.T3 = w.R3 + cc;
    w.Racc = w.T3 + cc;
    w.Rtmp = w.Racc + cc;
    w.L = w.Rtmp + cc;
    w.U = w.L + cc;
    w.V = w.U + cc;
    w.W = w.V + cc;
    w.US = w.W + cc;
    w.sig = w.US + cc;
    /* sig (c) | dinfo (8 doubles) | iinfo (32 ints): one d2h reads them all */
    w.dinfo = w.sig + c;
    w.iinfo = (int *)(w.dinfo + 8);
    w.cap = c;
    return w;
}

static step_ws get_ws(int c) { return get_ws_slot(c, PTT_WS_SMALL); }

static double tiny_pivot(void) { return 1.0e-14; }

/* Fukaya et al. shift for a Jacobi-scaled Gram of a len x c matrix. */
static double cholqr_shift(long len, int c) {
    double u = 0x1.0p-53;
    return 11.0 * ((double)len * c + (double)c * (c + 1)) * u * (double)c;
}

typedef struct {
    int deficient;
    double kappa;
    double maxdiag; /* largest diagonal entry of the Gram */
} chol_out;

static chol_out run_chol_k(int c, const double *G, double shift, double *R, double *T,
                           step_ws *w, int want_kappa) {
    chol_out o;
    ptt_hip_chol_qr_factor(c, G, shift, shift > 0 ? 0.0 : tiny_pivot(), R, T, w->iinfo, w->dinfo,
                           want_kappa);
    double kap[4] = {0.0, 0.0, 0.0, 0.0};
    ptt_hip_d2h(kap, w->dinfo, 4 * sizeof(double)); /* one transfer, waits for the kernel */
    o.deficient = (int)kap[2];
    o.maxdiag = kap[3];
    /* 2-norm estimate of the scaled factor (power iteration converges from
     * below; ||.||_F-condition / c is a guaranteed lower bound too) */
    o.kappa = kap[1] > kap[0] / c ? kap[1] : kap[0] / c;
    return o;
}

static chol_out run_chol(int c, const double *G, double shift, double *R, double *T, step_ws *w) {
    return run_chol_k(c, G, shift, R, T, w, 1);
}

/* Shifted factorization whose diagnostics are not needed: launched without
 * the condition estimate and without waiting for it (no host round trip). */
static void launch_chol_shifted(int c, const double *G, double shift, double *R, double *T,
                                step_ws *w) {
    ptt_hip_chol_qr_factor(c, G, shift, 0.0, R, T, w->iinfo, w->dinfo, 0);
}

/* In-place C = alpha * A * T (A: len x c, ld len; T c x c), A being core
 * `core` of x or, when buf is given, that buffer (c <= 128).  Uses the TMP
 * slot when the GEMM may not run in place (c > 128). */
static void apply_right(attac_tt *x, int core, double *buf, long len, int c, const double *T,
                        double alpha) {
    double *A = buf ? buf : x->coreList[core];
    if (c <= 128) {
        ptt_hip_dgemm('N', 'N', (int)len, c, c, alpha, A, len, T, c, 0.0, A, len);
    } else {
        double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)len * c);
        ptt_hip_dgemm('N', 'N', (int)len, c, c, alpha, A, len, T, c, 0.0, tmp, len);
        ptt_host_swap_core_with_tmp(x, core, len * c);
    }
}

/* In-place C = alpha * T^T * M (M: c x len, ld c; T c x c); M as in
 * apply_right. */
static void apply_left_t(attac_tt *x, int core, double *buf, int c, long len, const double *T,
                         double alpha) {
    double *M = buf ? buf : x->coreList[core];
    if (c <= 128) {
        ptt_hip_dgemm('T', 'N', c, (int)len, c, alpha, T, c, M, c, 0.0, M, c);
    } else {
        double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)len * c);
        ptt_hip_dgemm('T', 'N', c, (int)len, c, alpha, T, c, M, c, 0.0, tmp, c);
        ptt_host_swap_core_with_tmp(x, core, len * c);
    }
}

/* Q = A * T (A core `core`, len x c, c <= 128, in place) on the side stream:
 * the left-to-right sweep's next bond does not read core `core`, so forming Q
 * can run beside the next bond's one-workgroup Cholesky and its host round
 * trip.  The factorisation writes T straight into one of two side buffers
 * (side_tbuf: the main stream first waits for the side product that last
 * read it) or, in a rounding, into the core's own place (q_factor), which no
 * other bond writes.  The product is queued: side_flush launches it once the next
 * bond's Gram product is on the main stream (the side stream starts after
 * it), or at the end of the sweep, which then joins the side stream.  (A
 * rounding of d = 8, n = 1024, 128 columns of conditions 7 to 16: 6.60 ms with
 * these products on the main stream, 6.48 so.) */
static int g_side_parity = 0;
static struct {
    int pending, core, c, parity;
    long len;
    double alpha;
    attac_tt *x;
    double *tp;
} g_side_q;

static void side_flush(void) {
    if (!g_side_q.pending) return;
    g_side_q.pending = 0;
    ptt_hip_side_begin();
    ptt_hip_dgemm('N', 'N', (int)g_side_q.len, g_side_q.c, g_side_q.c, g_side_q.alpha,
                  g_side_q.x->coreList[g_side_q.core], g_side_q.len, g_side_q.tp, g_side_q.c,
                  0.0, g_side_q.x->coreList[g_side_q.core], g_side_q.len);
    ptt_hip_side_end(g_side_q.parity);
}

/* The side buffer the next factorisation writes T into (parity *p), once
 * the side product that last read it has finished. */
static double *side_tbuf(int *p) {
    double *ts = (double *)ptt_hip_scratch(PTT_WS_SIDE, sizeof(double) * 2 * 128 * 128);
    *p = g_side_parity;
    ptt_hip_side_wait(*p);
    return ts + (size_t)(*p) * 128 * 128;
}

/* tp: T, in side buffer p (from side_tbuf) or in the core's own place. */
static void apply_right_side(attac_tt *x, int core, long len, int c, double *tp, int p,
                             double alpha) {
    side_flush();
    g_side_parity = p ^ 1;
    g_side_q.pending = 1;
    g_side_q.x = x;
    g_side_q.core = core;
    g_side_q.len = len;
    g_side_q.c = c;
    g_side_q.alpha = alpha;
    g_side_q.parity = p;
    g_side_q.tp = tp;
}

/* ---- extreme magnitudes ---------------------------------------------------
 * Gram products and sums of squares square the entries: a carried core whose
 * entries lie below ~2^-450 (or above 2^450) would make them underflow
 * (overflow), and every pivot would die.  Such a core is scaled by an exact
 * power of two and the exponent is added to g_escale: the train then holds
 * 2^-g_escale times the input until the caller scales its result back, with
 * its tolerances scaled alike, so every decision and every value is the
 * unscaled computation's (powers of two are exact).  Callers reset g_escale
 * before their left-to-right sweep. */
static int g_escale = 0;
#define MAG_LO 0x1.0p-900
#define MAG_HI 0x1.0p+900

/* When sq (a Gram's largest diagonal entry or a sum of squares of the count
 * entries at p) lies outside [MAG_LO, MAG_HI], scale p by 2^-e, e the binary
 * exponent of max |p|, and return 1 (the caller recomputes); 0 otherwise,
 * also for an all-zero array. */
static int rescale_if_extreme(double *p, long count, double sq) {
    if (sq >= MAG_LO && sq <= MAG_HI) return 0;
    const double m = ptt_hip_maxabs(p, count);
    if (!(m > 0.0) || !(m < INFINITY)) return 0;
    const int e = ilogb(m);
    if (e == 0) return 0;
    ptt_hip_scale(p, count, ldexp(1.0, -e));
    g_escale += e;
    return 1;
}

/* Sum of squares of the last core after a left-to-right sweep, brought into
 * range by rescale_if_extreme (the core and g_escale change with it). */
static double last_core_sumsq(attac_tt *x) {
    int d = x->numDim;
    int rl = x->ttRank[d - 1];
    long cnt = (long)rl * x->dim[d - 1] * x->ttRank[d];
    double *dss = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 24;
    double ss = 0.0;
    for (int t = 0; t < 2; t++) {
        ptt_hip_sumsq(rl, x->dim[d - 1] * x->ttRank[d], x->coreList[d - 1], rl, dss);
        ptt_hip_d2h(&ss, dss, sizeof(double));
        if (!rescale_if_extreme(x->coreList[d - 1], cnt, ss)) break;
    }
    return ss;
}

/* Set while a left-to-right sweep may hand over to the Householder trees: a
 * core that one Cholesky-QR pass does not orthogonalise is left as it is and
 * the factorisation returns -1. */
static int g_one_pass_only = 0;
/* The last left-to-right sweep met a core (after core 0) of more than one pass. */
static int g_sweep_multi = 0;

/* Condition of the last factor up to which Q may be left unformed (below). */
#define KAPPA_UNFORMED 4.0

/* Set during a rounding: where core k's last factor T goes (c x c, NULL beyond 128
 * columns), and whether core k holds A with Q = qalpha A T left unformed.  The
 * right-to-left sweep multiplies core k by U Sigma of the bond after it, so A (T U
 * Sigma) takes one core-sized product instead of two: the last pass of a
 * factorisation left a write and a read of every core (95 us at 131072 x 128,
 * beside the main stream but on the same HBM and matrix cores) for a c x c by c x
 * rho product.  Both orders round to u times the condition of T, but not with the same
 * constant: at conditions up to 30 the cores of a rounding at n = 301, 59 columns were
 * 1.4 times as far from LAPACK's (2.8e-12 against 2.0e-12), so only a T of condition
 * at most KAPPA_UNFORMED is left. */
typedef struct {
    double *t, alpha;
    int unformed;
} q_factor;
static q_factor *g_qf = NULL;

/* Cholesky-QR of a core viewed as len x c (trans 'T': columns, LTR) or as
 * c x len (trans 'N': rows, RTL).  On return the core holds Q (alpha
 * applied) and R (c x c upper, A = Q*R resp. M = R^T*Q) is in *Rout.
 * Returns the number of passes. */
static int cholqr_core_g(attac_tt *x, int core, double *buf, char trans, long len, int c,
                         double qalpha, step_ws *w, const double **Rout, int allow_one_pass_noq,
                         int *one_pass, const double **T1out, int gram_ready);

static int cholqr_core(attac_tt *x, int core, double *buf, char trans, long len, int c,
                       double qalpha, step_ws *w, const double **Rout, int allow_one_pass_noq,
                       int *one_pass, const double **T1out) {
    return cholqr_core_g(x, core, buf, trans, len, c, qalpha, w, Rout, allow_one_pass_noq,
                         one_pass, T1out, 0);
}

/* gram_ready: w->G already holds the first pass's Gram. */
static int cholqr_core_g(attac_tt *x, int core, double *buf, char trans, long len, int c,
                         double qalpha, step_ws *w, const double **Rout, int allow_one_pass_noq,
                         int *one_pass, const double **T1out, int gram_ready) {
    double *A = buf ? buf : x->coreList[core];
    /* Mixed precision (left-to-right cores of up to 128 columns): the first
     * pass factors the Gram of the FP32-rounded core (FP32 MFMA, FP32
     * accumulation) and at least one FP64 pass follows, which restores FP64
     * orthogonality (mixed-precision CholeskyQR2: Yamazaki, Tomov and
     * Dongarra, SIAM J. Sci. Comput. 37, 2015). */
    const int leaf32 = g_leaf32 && trans == 'T' && !buf && c <= 128;
    q_factor *qf = (trans == 'T' && !buf && g_qf && g_qf[core].t) ? &g_qf[core] : NULL;
    /* a one-pass bond's Q may go to the side stream: T is then factored
     * straight into a side buffer, or stays where a rounding keeps it */
    const int side_q = trans == 'T' && !buf && c <= 128 && len * c >= (1L << 22) &&
                       ptt_hip_side_enabled();
    int side_p = g_side_parity;
    double *T1 = qf ? qf->t : side_q ? side_tbuf(&side_p) : w->T1;
    chol_out o;
    for (int t = 0; t < 2; t++) {
        if (t == 0 && gram_ready)
            ;
        else if (leaf32)
            ptt_hip_gram32(trans, c, len, A, len, w->G);
        else
            ptt_hip_gram(trans, c, len, A, trans == 'T' ? len : c, w->G);
        side_flush(); /* the previous bond's Q runs beside this factorisation */
        o = run_chol(c, w->G, 0.0, w->R1, T1, w);
        /* the carried core of the left-to-right sweep, brought into range */
        if (t > 0 || buf || trans != 'T' || !rescale_if_extreme(A, len * c, o.maxdiag)) break;
    }
    if (g_one_pass_only && !(o.deficient == 0 && o.kappa <= KAPPA_ONE_PASS)) return -1;
    if (!buf && trans == 'T' && core < 64) g_stats.kappa_ltr[core] = o.kappa;
    if (!buf && trans == 'N' && core < 64) g_stats.kappa_rtl[core] = o.kappa;
    if (one_pass) *one_pass = 0;
    if (!leaf32 && o.deficient == 0 && o.kappa <= KAPPA_ONE_PASS) {
        if (allow_one_pass_noq) {
            /* caller forms the new core itself from T1 (no explicit Q) */
            *Rout = w->R1;
            *T1out = T1;
            if (one_pass) *one_pass = 1;
            return 1;
        }
        /* small products gain less from the overlap than the copy of T and
         * the stream events cost */
        if (qf && o.kappa <= KAPPA_UNFORMED) {
            qf->alpha = qalpha;
            qf->unformed = 1;
        } else if (side_q)
            apply_right_side(x, core, len, c, T1, side_p, qalpha);
        else if (trans == 'T')
            apply_right(x, core, buf, len, c, T1, qalpha);
        else
            apply_left_t(x, core, buf, c, len, T1, qalpha);
        *Rout = w->R1;
        return 1;
    }
    /* Multi-pass Cholesky-QR that never drops content: a pass whose Gram is
     * deficient (a pivot below the guard) or too ill-conditioned is factored
     * with the Fukaya et al. shift instead.  A shifted pass still satisfies
     * A = Q R exactly and only leaves Q less orthogonal, so passes continue
     * until the last one started from a well-conditioned Q: two unshifted
     * passes after a shifted one, one after a moderately conditioned one,
     * at most CHOLQR_MAX_PASSES.  (Dropping a deficient pivot instead would
     * discard up to sqrt(guard) of that row's content.) */
    const double shift = cholqr_shift(len, c);
    int need;
    if (!(o.deficient == 0 && o.kappa <= KAPPA_TWO_PASS)) {
        launch_chol_shifted(c, w->G, shift, w->R1, T1, w);
        need = 2;
    } else {
        need = 1;
    }
    int passes = 1;
    /* pass 1 */
    if (trans == 'T') apply_right(x, core, buf, len, c, T1, 1.0);
    else apply_left_t(x, core, buf, c, len, T1, 1.0);
    /* the accumulated R: R1 after the first pass, then the product of every
     * pass's factor, alternating between two buffers (no copies) */
    double *Racc = w->R1;
    double *spare[2] = {w->Racc, w->Rtmp};
    int si = 0;
    while (need > 0) {
        passes++;
        A = buf ? buf : x->coreList[core];
        ptt_hip_gram(trans, c, len, A, trans == 'T' ? len : c, w->G);
        double *Rp = (passes % 2 == 0) ? w->R2 : w->R3;
        double *Tp = qf ? qf->t : (passes % 2 == 0) ? w->T2 : w->T3;
        chol_out q = run_chol(c, w->G, 0.0, Rp, Tp, w);
        if (q.deficient != 0 || q.kappa > KAPPA_TWO_PASS) {
            launch_chol_shifted(c, w->G, shift, Rp, Tp, w);
            need = 2;
        } else {
            need = (q.kappa <= KAPPA_ONE_PASS) ? 0 : 1;
        }
        if (passes >= CHOLQR_MAX_PASSES) need = 0;
        const double a = (need == 0) ? qalpha : 1.0;
        if (qf && need == 0 && q.deficient == 0 && q.kappa <= KAPPA_UNFORMED) {
            qf->alpha = qalpha;
            qf->unformed = 1;
        } else if (trans == 'T') apply_right(x, core, buf, len, c, Tp, a);
        else apply_left_t(x, core, buf, c, len, Tp, a);
        /* Racc <- Rp * Racc, into the buffer Racc does not occupy */
        double *out = spare[si];
        si ^= 1;
        ptt_hip_trmm_small(c, Rp, Racc, out);
        Racc = out;
    }
    *Rout = Racc;
    return passes;
}

/* Q = I_m (scaled) in core `core` viewed as m x m. */
static void set_identity(double *dst, int m, double alpha) {
    ptt_hip_zero(dst, sizeof(double) * (size_t)m * m);
    ptt_host_set_diag(dst, m, alpha);
}

/* Left-to-right sweep over cores 0..d-2.  qscale[k]: alpha of core k's Q;
 * rscale[k]: alpha applied when R_k multiplies core k+1.  With hand_over the
 * sweep stops before the first core after core 0 that needs more than one
 * Cholesky-QR pass.  Returns the cores left orthogonal (d - 1 if all). */
static int ltr_sweep_until(attac_tt *x, const double *qscale, const double *rscale,
                           int hand_over) {
    int d = x->numDim;
    int *r = x->ttRank, *n = x->dim;
    g_sweep_multi = 0;
    for (int i = 0; i < d - 1; i++) {
        long m = (long)r[i] * n[i];
        int c = r[i + 1];
        long wcols = (long)n[i + 1] * r[i + 2];
        if (m < c) {
            /* Q = I_m, R = A (m x c): core i+1 <- A * B (pattac.c:288's
             * rank rule r_{i+1} <- min(r_i n_i, r_{i+1})) */
            double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)m * wcols);
            ptt_hip_dgemm('N', 'N', (int)m, (int)wcols, c, rscale[i], x->coreList[i], m,
                          x->coreList[i + 1], c, 0.0, tmp, m);
            ptt_host_swap_core_with_tmp(x, i + 1, m * wcols);
            set_identity(x->coreList[i], (int)m, qscale[i]);
            r[i + 1] = (int)m;
            if (i < 64) g_stats.ltr_cholqr_passes[i] = 0;
            continue;
        }
        step_ws w = get_ws(c);
        const double *R = NULL;
        g_one_pass_only = hand_over && i > 0;
        int passes = cholqr_core(x, i, NULL, 'T', m, c, qscale[i], &w, &R, 0, NULL, NULL);
        g_one_pass_only = 0;
        if (passes < 0) {
            side_flush();
            ptt_hip_side_join();
            return i;
        }
        if (i < 64) g_stats.ltr_cholqr_passes[i] = passes;
        if (i > 0 && passes > 1) g_sweep_multi = 1;
        /* core i+1 (c x wcols) <- rscale * R * core i+1 */
        if (c <= 128) {
            ptt_hip_dgemm('N', 'N', c, (int)wcols, c, rscale[i], R, c, x->coreList[i + 1], c, 0.0,
                          x->coreList[i + 1], c);
        } else {
            double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)c * wcols);
            ptt_hip_dgemm('N', 'N', c, (int)wcols, c, rscale[i], R, c, x->coreList[i + 1], c, 0.0,
                          tmp, c);
            ptt_host_swap_core_with_tmp(x, i + 1, (long)c * wcols);
        }
    }
    side_flush();
    ptt_hip_side_join(); /* every Q formed on the side stream is in place */
    return d - 1;
}

static void ltr_sweep(attac_tt *x, const double *qscale, const double *rscale) {
    (void)ltr_sweep_until(x, qscale, rscale, 0);
}

/* Reference tail rule (pattac.c:468-481) on a descending list: the loop
 * accumulates sig_j^2 from the bottom and lowers rho while sqrt(sum) < delta.
 * tail0 is the energy beyond the list (0 for a full spectrum). */
static int tail_rule(const double *sig, int nsig, double tail0, double delta) {
    int rho = nsig;
    double sum = tail0;
    for (int j = nsig - 1; j >= 0; j--) {
        sum += sig[j] * sig[j];
        if (sqrt(sum) < delta) rho = j;
        else break;
    }
    return rho;
}

/* Columns beyond which the SVD of a bond with more rows than columns starts from the
 * eigenvectors of the small Gram. */
#define TALL_WARM_MIN 32

/* Robust right-to-left step: explicit LQ by (shifted) Cholesky-QR, SVD of
 * L, new core = V_rho^T Q.  Up to 128 rows the SVD pivots L's columns itself and
 * gives the right vectors alone: U Sigma = L V.  Beyond (and where the whole
 * spectrum is wanted, noise included) the rows of M are first put
 * in order of decreasing norm (the Gram's diagonal), so that the columns of
 * L come by decreasing norm: Drmac and Veselic's diagonal pivoting (SIAM J.
 * Matrix Anal. Appl. 29, 2008), applied statically as on the Gram route,
 * which cuts the Jacobi sweeps on graded bonds.  With P M = L Q and L =
 * U Sigma V^T, M = (P^T U) Sigma (V^T Q): the new core is unchanged and only
 * the rows of U Sigma are put back.
 * warm: the Gram route has just refused the bond and left its Gram in ws->G and
 * its vectors U in ws->V, which resolve every direction: the Jacobi starts from
 * R U, at any number of rows the Gram route takes. */
static int rtl_step_robust(attac_tt *x, int i, const int *maxr, double delta,
                           const double *nscale, step_ws *ws, int *passes_out, int warm) {
    int *r = x->ttRank, *n = x->dim;
    int rows = r[i];
    long w = (long)n[i] * r[i + 1];
    const double *R = NULL, *T1 = NULL;
    int one_pass = 0;
    if (g_whole_spectra) warm = 0;
    const int right = (rows <= 128 || warm) && !g_whole_spectra;
    const int sorted = !right && rows >= 8 && rows <= 1024;
    int *perm = (int *)ws->W; /* W is free on this route */
    if (sorted) {
        double *M = x->coreList[i];
        ptt_hip_gram('N', rows, w, M, rows, ws->T3);
        ptt_hip_sym_sort_perm(rows, ws->T3, ws->G, perm); /* G = P G P^T, the Gram of P M */
        double *t2 = (double *)ptt_hip_scratch(PTT_WS_TMP2, sizeof(double) * (size_t)rows * w);
        ptt_hip_permute_rows(rows, (int)w, perm, M, rows, t2, rows);
        ptt_hip_d2d(M, t2, sizeof(double) * (size_t)rows * w);
    }
    int passes = cholqr_core_g(x, i, NULL, 'N', w, rows, 1.0, ws, &R, 0, &one_pass, &T1,
                               sorted || warm);
    *passes_out = passes;
    if (warm) {
        ptt_hip_svd_right_from(rows, R, rows, ws->V, rows, ws->U, ws->sig, ws->V, rows, delta,
                               maxr[i], ws->iinfo + 1);
    } else if (right) {
        ptt_hip_svd_right(rows, R, rows, ws->U, ws->sig, ws->V, rows, delta, maxr[i],
                          ws->iinfo + 1);
    } else {
        ptt_hip_transpose(rows, rows, R, rows, ws->L, rows, 1.0);
        ptt_hip_svd_jacobi(rows, rows, ws->L, rows, ws->sig, ws->U, rows, ws->V, rows, 0.0, delta,
                           maxr[i], ws->iinfo + 1);
    }
    /* sigma, factor info and SVD info are contiguous: one transfer */
    const size_t nb = sizeof(double) * ((size_t)rows + 8) + sizeof(int) * 8;
    double *hb = (double *)ptt_host_malloc(nb);
    ptt_hip_d2h(hb, ws->sig, nb);
    keep_hsig(hb, rows);
    int io[3];
    memcpy(io, (const int *)(hb + rows + 8) + 1, sizeof io);
    free(hb);
    int rho = io[1];
    if (i < 64) { g_stats.svd_sweeps[i] = io[2]; g_stats.numrank[i] = io[0]; }
    double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)rho * w);
    double *us = sorted ? ws->L : ws->US;
    if (right)
        ptt_hip_dgemm('T', 'N', rows, rho, rows, 1.0, R, rows, ws->V, rows, 0.0, us, rows);
    else
        ptt_hip_svd_factors(rows, rho, ws->iinfo + 2, ws->U, rows, ws->sig, 1.0, NULL, us);
    if (sorted) ptt_hip_unpermute_rows(rows, rho, perm, us, rows, ws->US, rows);
    ptt_hip_dgemm('T', 'N', rho, (int)w, rows, nscale[i], ws->V, rows, x->coreList[i], rows, 0.0,
                  tmp, rho);
    ptt_host_swap_core_with_tmp(x, i, (long)rho * w);
    return rho;
}

/* Fast right-to-left step for a core whose kept directions are well
 * conditioned: Gram -> eigen-decomposition (U, Sigma) -> new core =
 * Sigma^-1 U^T M in one GEMM.  The discarded energy is measured from the
 * explicit residual M - U Sigma (new core), accurate to rounding of M
 * itself, so the tail rule is decided exactly as with an orthogonal LQ;
 * the residual is skipped when the trace alone shows that the cap binds.
 * Returns rho, or a negative value when the step must be redone by the
 * robust path (the core is left unchanged in that case; -3: ws->G and ws->V
 * hold its Gram and vectors that resolve every direction). */
/* Accuracy of the Gram route against an orthogonal (LQ) factorization for a
 * cut after rho of the rows singular values sig (descending): the Gram's
 * rounding, ~ rows*u*s0^2, turns the kept subspace by about
 * est = rows*u*s0^2 / (s_{rho-1}^2 - s_rho^2) (when nothing is cut, est is
 * the new rows' loss of orthonormality), which exceeds the LQ route's
 * rows*u*s0 / (s_{rho-1} - s_rho) by the factor s0 / (s_{rho-1} + s_rho).
 * The Gram route is kept only when est is negligible or that factor is at
 * most 2, so its result stays as close to the reference's orthogonal
 * rounding as the problem's own sensitivity allows.  `dropped` is the
 * squared content set to zero before the small SVD or eigen-decomposition,
 * added to the Gram's rounding. */
static int gram_route_accurate(const double *sig, int rows, int rho, double dropped) {
    const double s0 = sig[0], sl = sig[rho - 1], sn = (rho < rows) ? sig[rho] : 0.0;
    const double gap2 = (sl - sn) * (sl + sn);
    if (!(s0 > 0.0) || !(gap2 > 0.0)) return 0;
    const double est = (rows * 0x1.0p-53 * s0 * s0 + dropped) / gap2;
    return est <= FAST_EST_MAX || s0 <= 2.0 * (sl + sn);
}

/* The Gram route's small dense problem: the eigen-decomposition of the
 * Gram by tridiagonalisation and divide and conquer (default), or, with
 * PARATT_AMD_GRAM_JACOBI=1 in the environment, the one-sided Jacobi SVD of
 * its diagonally pivoted Cholesky factor. */
static int gram_use_eig(void) {
    static int v = -1;
    if (v < 0) {
        const char *e = getenv("PARATT_AMD_GRAM_JACOBI");
        v = !(e && e[0] == '1');
    }
    return v;
}

/* The new core of a right-to-left Gram-route step whose rank the cap
 * decides, W M (W = scaled Sigma^-1 U^T, rho x rows), on the side stream:
 * the sweep's next bond reads core i-1 and U Sigma only.  The product is
 * queued once the next bond's Gram is on the main stream (rside_flush), so
 * it runs beside that bond's one-workgroup eigensolver rather than its
 * full-GPU products.  W is formed in one of two side buffers (the main
 * stream first waits for the side product that last read it); the product
 * writes one of two pool buffers, which core i takes at once while the pool
 * takes core i's old buffer: that buffer is read by the pending product and
 * written only by a later side product (the same stream, in order) or freed
 * by a growth, which waits for both streams.  rtl_sweep flushes and joins
 * the side stream at its end. */
static int g_rside_parity = 0, g_rside_used = 0;
static struct {
    int pending, p, rho, rows;
    long w;
    const double *W, *M;
    double *B;
} g_rq;

static void rside_flush(void) {
    if (!g_rq.pending) return;
    g_rq.pending = 0;
    ptt_hip_side_begin();
    ptt_hip_dgemm('N', 'N', g_rq.rho, (int)g_rq.w, g_rq.rows, 1.0, g_rq.W, g_rq.rho, g_rq.M,
                  g_rq.rows, 0.0, g_rq.B, g_rq.rho);
    ptt_hip_side_end(g_rq.p);
    g_rside_used = 1;
}

static int rtl_step_fast(attac_tt *x, int i, const int *maxr, double delta,
                         const double *nscale, step_ws *ws) {
    int *r = x->ttRank, *n = x->dim;
    int rows = r[i];
    long w = (long)n[i] * r[i + 1];
    double *M = x->coreList[i];
    /* beyond 1024 rows the orthogonal route handles the bond */
    if (rows > 1024) return -1;
    ptt_hip_gram('N', rows, w, M, rows, ws->G);
    rside_flush(); /* the previous bond's new core beside this bond's eigensolver */
    const int eig = (rows <= 192) && gram_use_eig();
    int *cidx = (int *)ws->Rtmp;
    if (eig) {
        /* G = U diag(sig^2) U^T; eigenvalues below the Gram's own rounding
         * (FAST_DROP * rows * u * lambda_max in total) are set to zero. */
        ptt_hip_syev_gram(rows, ws->G, ws->sig, ws->V, rows, cidx, ws->iinfo + 1, ws->dinfo,
                          delta, maxr[i], FAST_DROP * rows * 0x1.0p-53);
    } else {
        /* Factor the Gram with its indices ordered by decreasing diagonal:
         * the columns of L = R^T then come by decreasing norm, which roughly
         * halves the Jacobi sweeps on graded bond spectra.  L's rows are in
         * that order, so U's rows are put back afterwards. */
        ptt_hip_sym_sort_perm(rows, ws->G, ws->T2, cidx);
        ptt_hip_chol_qr_factor(rows, ws->T2, 0.0, tiny_pivot(), ws->R1, NULL, ws->iinfo,
                               ws->dinfo, 0);
        ptt_hip_transpose(rows, rows, ws->R1, rows, ws->L, rows, 1.0);
        /* Columns of L whose squared norms together stay below the Gram's
         * own rounding (FAST_DROP * rows * u * max norm^2) carry no
         * information this route can resolve: zeroed, they take no part in
         * the rotations. */
        ptt_hip_drop_small_cols(rows, rows, ws->L, rows, FAST_DROP * rows * 0x1.0p-53,
                                ws->dinfo + 5);
        ptt_hip_svd_jacobi(rows, rows, ws->L, rows, ws->sig, ws->U, rows, NULL, rows, 0.0, delta,
                           maxr[i], ws->iinfo + 1);
        ptt_hip_unpermute_rows(rows, rows, cidx, ws->U, rows, ws->V, rows);
    }
    /* sigma, factor info and SVD info are contiguous: one transfer.  On the
     * Gram route the factors for the rank the cap gives (the rank whenever
     * the spectrum holds that many values above the noise), and the new core
     * unless it may go to the side stream, are queued behind the copy, so
     * they run while the host reads sigma and decides; another rank launches
     * them again below. */
    size_t nb = sizeof(double) * ((size_t)rows + 8) + sizeof(int) * 8;
    double *hb = (double *)ptt_host_malloc(nb);
    const unsigned long long tk = ptt_hip_d2h_begin(ws->sig, nb);
    const int spec = eig ? (maxr[i] < rows ? maxr[i] : rows) : 0;
    /* the new core may go to the side stream (decided once sigma is read) */
    const int side_ok = spec > 0 && rows <= 128 && x->coreMem != NULL && ptt_hip_side_enabled() &&
                        (double)spec * rows * (double)w >= 0x1.0p28;
    const int sp = g_rside_parity;
    double *Wspec = ws->W;
    double *tmp = NULL;
    if (spec > 0) {
        if (side_ok) {
            Wspec = (double *)ptt_hip_scratch(PTT_WS_RSIDE, sizeof(double) * 2 * 128 * 128) +
                    (size_t)sp * 128 * 128;
            ptt_hip_side_wait(sp);
        }
        ptt_hip_svd_factors_perm(rows, spec, cidx, ws->V, rows, ws->sig, nscale[i], Wspec,
                                 ws->US);
        if (!side_ok) {
            tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)spec * w);
            ptt_hip_dgemm('N', 'N', spec, (int)w, rows, 1.0, Wspec, spec, M, rows, 0.0, tmp,
                          spec);
        }
    }
    ptt_hip_d2h_end(tk, hb, nb);
    double *sig = hb;
    const int *io = (const int *)(hb + rows + 8) + 1;
    int numrank = io[0];
    if (i < 64) { g_stats.svd_sweeps[i] = io[2]; g_stats.numrank[i] = numrank; }
    /* refused: -3 when the vectors in ws->V resolve every direction */
    const int refused = (eig && numrank == rows) ? -3 : -2;
    int cap = maxr[i] < rows ? maxr[i] : rows;
    int rho0 = cap < numrank ? cap : numrank;
    if (rho0 < 1) rho0 = 1;
    const double s0 = sig[0];
    /* statistics: condition of the kept directions */
    if (i < 64) g_stats.kappa_rtl[i] = sig[rho0 - 1] > 0.0 ? s0 / sig[rho0 - 1] : 0.0;
    if (!(s0 > 0.0)) { free(hb); return -1; }
    /* The Gram's squared singular values carry an absolute error below
     * floor2 (a wide margin over rows*u*s0^2).  When the cap binds and the
     * last kept value squared exceeds delta^2 by more than that error, the
     * rule's tail from rho0-1 (which holds sigma_{rho0-1}^2) exceeds delta^2
     * whatever lies beyond the list: the rank is the cap and the energy
     * beyond the list is not needed. */
    const double floor2 = 1e4 * rows * 0x1.0p-53 * s0 * s0;
    const double sl2 = sig[rho0 - 1] * sig[rho0 - 1];
    const int cut_at_cap = (rho0 == cap) && (sl2 - floor2 >= delta * delta);
    if (side_ok && rho0 == spec && cut_at_cap) {
        if (!gram_route_accurate(sig, rows, rho0, hb[rows + 5])) {
            free(hb);
            return refused;
        }
        g_rside_parity ^= 1;
        double *B = (double *)ptt_hip_scratch(PTT_WS_ROUT0 + sp,
                                              sizeof(double) * (size_t)rho0 * w);
        g_rq.pending = 1;
        g_rq.p = sp;
        g_rq.rho = rho0;
        g_rq.rows = rows;
        g_rq.w = w;
        g_rq.W = Wspec;
        g_rq.M = M;
        g_rq.B = B;
        size_t capb = (size_t)x->coreMem[i] * sizeof(double);
        ptt_hip_swap_tmp(PTT_WS_ROUT0 + sp, &x->coreList[i], &capb);
        size_t el = capb / sizeof(double);
        x->coreMem[i] = (int)(el > 2147483647UL ? 2147483647UL : el);
        keep_hsig(sig, rows);
        free(hb);
        return rho0;
    }
    if (rho0 == spec && side_ok) {
        /* W is in the side buffer; the product runs here */
        tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)spec * w);
        ptt_hip_dgemm('N', 'N', spec, (int)w, rows, 1.0, Wspec, spec, M, rows, 0.0, tmp, spec);
    }
    if (rho0 != spec) {
        tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)rho0 * w);
        if (eig)
            ptt_hip_svd_factors_perm(rows, rho0, cidx, ws->V, rows, ws->sig, nscale[i], ws->W,
                                     ws->US);
        else
            ptt_hip_svd_factors(rows, rho0, NULL, ws->V, rows, ws->sig, nscale[i], ws->W, ws->US);
        ptt_hip_dgemm('N', 'N', rho0, (int)w, rows, 1.0, ws->W, rho0, M, rows, 0.0, tmp, rho0);
    }
    /* Otherwise the energy beyond the kept list.  When the cap binds and the
     * trace of the Gram minus the kept squared values exceeds delta^2 by more
     * than their rounding, the rule keeps the cap and no residual is needed;
     * otherwise the residual M - U Sigma (new core)/sqrt(n_i) is formed out
     * of place (M stays untouched) and its Frobenius norm gives the tail
     * exactly. */
    double tail2 = -1.0;
    if (!cut_at_cap && eig && rho0 == cap) {
        double kept = 0.0;
        for (int q = 0; q < rho0; q++) kept += sig[q] * sig[q];
        const double trace = hb[rows + 7];
        const double err = 64.0 * rows * 0x1.0p-53 * trace;
        if (trace - kept - err >= delta * delta && trace - kept - err > 0.0) tail2 = trace - kept;
    }
    if (!cut_at_cap && tail2 < 0.0) {
        double *E = (double *)ptt_hip_scratch(PTT_WS_RES, sizeof(double) * (size_t)rows * w);
        ptt_hip_d2d(E, M, sizeof(double) * (size_t)rows * w);
        ptt_hip_dgemm('N', 'N', rows, (int)w, rho0, -1.0 / nscale[i], ws->US, rows, tmp, rho0,
                      1.0, E, rows);
        double *dss = ws->dinfo + 4;
        ptt_hip_sumsq(rows, (int)w, E, rows, dss);
        ptt_hip_d2h(&tail2, dss, sizeof(double));
    }
    int rho = rho0;
    int trust;
    if (cut_at_cap) {
        trust = 1;
    } else if (sqrt(tail2) >= delta) {
        /* the tail beyond the kept list is too large: that is the answer only
         * when the cap binds.  Otherwise the exact rounding keeps directions
         * below the Gram's resolution, which this step cannot resolve. */
        trust = (rho0 == cap);
    } else {
        /* The tail beyond the kept list is below delta, so the cut may move
         * inside the list: the rule's walk is reliable when delta^2 is far
         * above the Gram's error floor2, and the cut certainly stays at rho0
         * when the last kept value squared exceeds delta^2 by more than that
         * error (tail_{rho0-1}^2 = tail2 + s_{rho0-1}^2 >= delta^2). */
        if (!(delta * delta < floor2)) {
            trust = 1;
            rho = tail_rule(sig, rho0, tail2, delta);
            if (rho < 1) rho = 1;
        } else {
            trust = (sl2 - floor2 >= delta * delta);
        }
    }
    if (trust) trust = gram_route_accurate(sig, rows, rho, hb[rows + 5]);
    if (!trust) {
        free(hb);
        return refused;
    }
    if (rho < rho0) {
        /* keep the first rho rows of the new core and the first rho columns of U Sigma */
        double *t2 = (double *)ptt_hip_scratch(PTT_WS_TMP2, sizeof(double) * (size_t)rho * w);
        ptt_hip_copy2d(rho, (int)w, tmp, rho0, t2, rho, 1.0);
        ptt_hip_d2d(tmp, t2, sizeof(double) * (size_t)rho * w);
    }
    ptt_host_swap_core_with_tmp(x, i, (long)rho * w);
    keep_hsig(sig, rows);
    free(hb);
    return rho;
}

/* Sketched right-to-left step: a randomized range finder (Halko, Martinsson
 * and Tropp, SIAM Review 2011, Alg. 4.4: Gaussian test matrix, one power
 * iteration) with l = predicted rank + oversampling columns replaces the
 * rows x rows factorization and SVD of the plain step by l x l ones.
 *
 * Certification (the rank must equal the plain method's): with Q the
 * orthonormal sketch basis, B = Q^T M and sigma^_j its singular values,
 * sigma^_j <= sigma_j (interlacing), and the exact residual energy
 * e2 = ||M - Q B||^2 satisfies e2 + sum_{q>=j, q<l} sigma^_q^2
 * >= sum_{q>=j} sigma_q^2 = tail_j^2.  The candidate rank rho (the tail rule
 * on the sketch with e2 added) thus has tail_rho < delta, so the plain rank
 * is <= rho; and if sigma^_{rho-1} >= delta then tail_{rho-1} >= delta, so
 * the plain rank is >= rho.  Anything else -- the residual alone above
 * delta, the lower bound failing, or the cap binding (where the truncation
 * error is not eps-controlled) -- returns -1 and the plain step runs on the
 * untouched core.  On acceptance the new core is V_rho^T Q_B (orthonormal
 * rows) and ws->US = Q U_rho Sigma_rho, as in the plain steps. */
static int rtl_step_sketch(attac_tt *x, int i, const int *maxr, double delta,
                           const double *nscale, step_ws *ws, int l) {
    int *r = x->ttRank, *n = x->dim;
    const int rows = r[i];
    const long w = (long)n[i] * r[i + 1];
    double *M = x->coreList[i];
    const size_t need = (size_t)w * l + 2 * (size_t)rows * l + (size_t)l * w +
                        (size_t)rows * w + (size_t)l * l;
    double *Om = (double *)ptt_hip_scratch(PTT_WS_RSK, sizeof(double) * need);
    double *Y = Om + (size_t)w * l;       /* rows x l: sketch, then basis Q */
    double *QL = Y + (size_t)rows * l;    /* rows x l */
    double *B = QL + (size_t)rows * l;    /* l x w */
    double *E = B + (size_t)l * w;        /* rows x w: residual */
    double *USB = E + (size_t)rows * w;   /* l x l */
    step_ws sw = get_ws_slot(l, PTT_WS_SMALL2);
    const double *R = NULL;
    ptt_hip_gauss_fill(Om, w * l, g_sketch_seed++, 0, 1.0);
    ptt_hip_dgemm('N', 'N', rows, l, (int)w, 1.0, M, rows, Om, w, 0.0, Y, rows);
    cholqr_core(NULL, 0, Y, 'T', rows, l, 1.0, &sw, &R, 0, NULL, NULL);
    /* one power iteration: Y <- M (M^T Q) */
    ptt_hip_dgemm('T', 'N', (int)w, l, rows, 1.0, M, rows, Y, rows, 0.0, Om, w);
    ptt_hip_dgemm('N', 'N', rows, l, (int)w, 1.0, M, rows, Om, w, 0.0, Y, rows);
    cholqr_core(NULL, 0, Y, 'T', rows, l, 1.0, &sw, &R, 0, NULL, NULL);
    /* B = Q^T M = L_B Q_B (LQ by Cholesky-QR of the rows) */
    ptt_hip_dgemm('T', 'N', l, (int)w, rows, 1.0, Y, rows, M, rows, 0.0, B, l);
    cholqr_core(NULL, 0, B, 'N', w, l, 1.0, &sw, &R, 0, NULL, NULL);
    ptt_hip_transpose(l, l, R, l, sw.L, l, 1.0);
    /* residual of the rank-l approximation Q L_B Q_B, exact energy */
    ptt_hip_dgemm('N', 'N', rows, l, l, 1.0, Y, rows, sw.L, l, 0.0, QL, rows);
    ptt_hip_d2d(E, M, sizeof(double) * (size_t)rows * w);
    ptt_hip_dgemm('N', 'N', rows, (int)w, l, -1.0, QL, rows, B, l, 1.0, E, rows);
    ptt_hip_sumsq(rows, (int)w, E, rows, sw.dinfo + 4);
    ptt_hip_svd_jacobi(l, l, sw.L, l, sw.sig, sw.U, l, sw.V, l, 0.0, delta, l, sw.iinfo + 1);
    double *hb = (double *)ptt_host_malloc(sizeof(double) * ((size_t)l + 8));
    ptt_hip_d2h(hb, sw.sig, sizeof(double) * ((size_t)l + 8));
    const double e2 = hb[l + 4];
    int rho = -1;
    if (sqrt(e2) < delta) {
        int rs = tail_rule(hb, l, e2, delta);
        const int cap = maxr[i] < rows ? maxr[i] : rows;
        int ok = (rs <= cap) && (rs == 0 || hb[rs - 1] >= delta);
        if (ok) rho = rs < 1 ? 1 : rs;
    }
    if (rho > 0) {
        int h_rho = rho;
        ptt_hip_h2d_queued(sw.iinfo + 8, &h_rho, sizeof(int));
        /* new core (rho x w) = sqrt(n_i) V_rho^T Q_B */
        double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)rho * w);
        ptt_hip_dgemm('T', 'N', rho, (int)w, l, nscale[i], sw.V, l, B, l, 0.0, tmp, rho);
        ptt_host_swap_core_with_tmp(x, i, (long)rho * w);
        /* U Sigma of the bond: Q (U_B Sigma)_rho */
        ptt_hip_svd_factors(l, rho, sw.iinfo + 8, sw.U, l, sw.sig, 1.0, NULL, USB);
        ptt_hip_dgemm('N', 'N', rows, rho, l, 1.0, Y, rows, USB, l, 0.0, ws->US, rows);
        ptt_hip_d2d(ws->sig, sw.sig, sizeof(double) * (size_t)l);
    }
    free(hb);
    return rho;
}

/* Columns of the sketch that pred allows for bond i of rows x w; 0: none. */
static int sketch_columns(const int *pred, int i, int rows, long w) {
    if (i >= 64 || pred[i] <= 0 || pred[i] > 128 - SKETCH_OVERSAMPLE) return 0;
    const int l = pred[i] + SKETCH_OVERSAMPLE;
    return (2 * l <= rows && (long)l <= w) ? l : 0;
}

/* Right-to-left truncation (pattac.c:297-522) of a left-orthogonal TT whose
 * cores carry the reference's scaled magnitudes; tol is absolute in that
 * scaled space.  nscale[k] = sqrt(n_k) is applied to each finished core. */
static void rtl_sweep(attac_tt *x, const int *maxr, double abs_tol, const double *nscale) {
    int d = x->numDim;
    int *r = x->ttRank, *n = x->dim;
    const double delta = (d > 1) ? abs_tol / sqrt(d - 1.0) : abs_tol;
    int prev_robust = 0;
    for (int i = d - 1; i > 0; i--) {
        int rows = r[i];
        long w = (long)n[i] * r[i + 1];
        long m1 = (long)r[i - 1] * n[i - 1];
        g_hsig_n = 0;
        double left_alpha = (i == 1) ? nscale[0] : 1.0;
        int cap = maxr[i];
        int rho;
        step_ws ws;
        /* a pending side product waits for the Gram-route step's Gram; any
         * other step queues it first */
        if (w < rows || prev_robust || g_pred) rside_flush();
        if (w < rows) {
            /* L has only w columns: SVD of the core itself (M = L*Q with Q = I_w) */
            int k = (int)w;
            ws = get_ws(rows > k ? rows : k);
            if (k > TALL_WARM_MIN && k <= 192 && !g_whole_spectra && gram_use_eig()) {
                /* The rotations start from M V0, V0 the eigenvectors of M^T M: its
                 * columns are nearly orthogonal (any orthogonal V0 gives the same
                 * result in more sweeps), and V = V0 times what they accumulate. */
                ptt_hip_gram('T', k, rows, x->coreList[i], rows, ws.G);
                ptt_hip_syev_gram(k, ws.G, ws.sig, ws.T1, k, (int *)ws.Rtmp, ws.iinfo + 1,
                                  ws.dinfo, 0.0, k, 0.0);
                ptt_hip_dgemm('N', 'N', rows, k, k, 1.0, x->coreList[i], rows, ws.T1, k, 0.0, ws.L,
                              rows);
                ptt_hip_svd_jacobi(rows, k, ws.L, rows, ws.sig, ws.U, rows, ws.T2, k, 0.0, delta,
                                   cap, ws.iinfo + 1);
                ptt_hip_dgemm('N', 'N', k, k, k, 1.0, ws.T1, k, ws.T2, k, 0.0, ws.V, k);
            } else {
                ptt_hip_svd_jacobi(rows, k, x->coreList[i], rows, ws.sig, ws.U, rows, ws.V, k, 0.0,
                                   delta, cap, ws.iinfo + 1);
            }
            int io[3];
            ptt_hip_d2h(io, ws.iinfo + 1, sizeof(int) * 3);
            g_hsig_n = 0;
            rho = io[1];
            if (i < 64) { g_stats.svd_sweeps[i] = io[2]; g_stats.numrank[i] = io[0]; g_stats.rtl_cholqr_passes[i] = 0; }
            /* core i <- sqrt(n_i) * V_rho^T (rho x w) */
            ptt_hip_transpose(k, rho, ws.V, k, x->coreList[i], rho, nscale[i]);
            ptt_hip_svd_factors(rows, rho, ws.iinfo + 2, ws.U, rows, ws.sig, 1.0, NULL, ws.US);
        } else {
            ws = get_ws(rows);
            int sk = -1;
            const int l = g_pred ? sketch_columns(g_pred, i, rows, w) : 0;
            if (l > 0) {
                g_sketch_counts[0]++;
                sk = rtl_step_sketch(x, i, maxr, delta, nscale, &ws, l);
                if (sk > 0) g_sketch_counts[1]++;
            }
            /* Bond spectra change slowly along the train: once the Gram
             * route was rejected at the right neighbour, go straight to the
             * orthogonal route (saves a Gram, a factorization and an SVD). */
            rho = (sk > 0) ? sk : prev_robust ? -1 : rtl_step_fast(x, i, maxr, delta, nscale, &ws);
            if (i < 64) g_stats.rtl_cholqr_passes[i] = (sk > 0) ? 20 : 1;
            if (i < 64) g_spec[i][19] = (sk > 0) ? 1.0 : 0.0;
            prev_robust = (rho < 0);
            if (rho < 0) {
                const int warm = (rho == -3);
                int passes = 0;
                rho = rtl_step_robust(x, i, maxr, delta, nscale, &ws, &passes, warm);
                if (i < 64) g_stats.rtl_cholqr_passes[i] = 10 + passes;
                /* a well-conditioned bond lets the next one try the Gram route */
                if (i < 64 && g_stats.kappa_rtl[i] <= 1.0e2) prev_robust = 0;
            }
        }
        if (i < 64) {
            /* the leading spectrum up to rho+3 in one transfer: the values
             * around the cut for the statistics and the spectrum record */
            double sv[132];
            int k = (int)(w < rows ? w : rows);
            /* sketch: the l Ritz values (lower bounds of the spectrum) */
            if (g_spec[i][19] != 0.0 && g_pred) k = g_pred[i] + SKETCH_OVERSAMPLE;
            int cnt = rho + 3 < k ? rho + 3 : k;
            if (cnt > 128) cnt = 128;
            if (g_spec[i][19] == 0.0 && g_hsig_n >= cnt)
                memcpy(sv, g_hsig, sizeof(double) * (size_t)cnt);
            else if (cnt > 0)
                ptt_hip_d2h(sv, ws.sig, sizeof(double) * cnt);
            for (int q = 0; q < 4; q++) {
                int j = rho - 1 + q;
                g_stats.sig[i][q] = (j >= 0 && j < cnt) ? sv[j] : 0.0;
            }
            for (int q = 0; q < 16; q++) {
                int j = rho - 13 + q;
                g_spec[i][q] = (j >= 0 && j < cnt) ? sv[j] : 0.0;
            }
            g_spec[i][16] = cnt > 0 ? sv[0] : 0.0;
            g_spec[i][17] = rho;
            g_spec[i][18] = rows;
        }
        /* core i-1 (m1 x rows) <- left_alpha * core i-1 * U_rho Sigma_rho */
        if (g_qf && g_qf[i - 1].unformed) {
            ptt_hip_dgemm('N', 'N', rows, rho, rows, g_qf[i - 1].alpha, g_qf[i - 1].t, rows, ws.US,
                          rows, 0.0, ws.U, rows);
            ws.US = ws.U;
            g_qf[i - 1].unformed = 0;
        }
        if (rho <= 128) {
            ptt_hip_dgemm('N', 'N', (int)m1, rho, rows, left_alpha, x->coreList[i - 1], m1, ws.US,
                          rows, 0.0, x->coreList[i - 1], m1);
        } else {
            double *tmp = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)m1 * rho);
            ptt_hip_dgemm('N', 'N', (int)m1, rho, rows, left_alpha, x->coreList[i - 1], m1, ws.US,
                          rows, 0.0, tmp, m1);
            ptt_host_swap_core_with_tmp(x, i - 1, m1 * rho);
        }
        r[i] = rho;
    }
    rside_flush();
    if (g_rside_used) {
        ptt_hip_side_join(); /* every new core formed on the side stream is in place */
        g_rside_used = 0;
    }
}

static void fill_scales(const attac_tt *x, double *inv, double *sq) {
    for (int k = 0; k < x->numDim; k++) {
        sq[k] = sqrt((double)x->dim[k]);
        inv[k] = 1.0 / sq[k];
    }
}

/* ---- low-rank trains ---------------------------------------------------------
 * Trains whose bond ranks are all at most TREE_RANK are rounded by Householder
 * trees (tsqr.hip) with every rank decided and kept on the device: a fixed
 * sequence of launches, one host read between the sweeps (the norm sets the
 * tolerance) and one at the end (ranks and singular values).  The left-to-right
 * sweep keeps each core's reflectors in place instead of forming Q; the
 * right-to-left sweep applies them to U Sigma of the bond before.  Accuracy is
 * that of an orthogonal factorisation at every bond, as on the LQ route.
 * The lines: above 32 columns a block of 512 rows no longer fits a workgroup's
 * registers.  From 17 to 32 the trees (255 us a bond at 22 columns, n = 83; 350
 * at 32, n = 32) lose to the Gram route on well-conditioned trains (211, 266
 * us), which take one Cholesky-QR pass and no Jacobi sweeps, and win on
 * ill-conditioned ones (some 600 us a bond there: three to four passes a
 * factorisation): such a train starts on the Cholesky-QR sweep and changes over
 * at the first core after core 0 that one pass does not orthogonalise.  So does one
 * with an unfolding of 11 to 16 columns and 8192 rows or more, whose blocks fill
 * the GPU less well than a Gram's (d = 8, us, trees / this way; before the trees):
 * 16 columns, n = 2048, well-conditioned 1401 / 848 (1129), deficient 1210 / 1331
 * (2250); 12 columns, n = 2048, 1135 / 802 (1046) and 1038 / 1150 (2083).  With
 * fewer rows or columns the trees lose nothing to the sweep they replaced. */
#define TREE_RANK_ALWAYS 16
#define TREE_RANK_TALL 10
#define TREE_ROWS_TALL 8192
#define TREE_RANK 32
#define TREE_ROWS 65536
/* 0: not by trees; 1: by trees; 2: by trees once a core is ill-conditioned. */
static int tree_route(const attac_tt *x) {
    const int d = x->numDim;
    int route = 1;
    if (d < 2 || g_leaf32 || g_pred || g_whole_spectra) return 0;
    for (int k = 0; k < d; k++) {
        const int r0 = x->ttRank[k], r1 = x->ttRank[k + 1];
        if (r0 < 1 || r1 < 1 || (k > 0 && r0 > TREE_RANK)) return 0;
        if (k > 0 && r0 > TREE_RANK_ALWAYS) route = 2;
        if ((r1 > TREE_RANK_TALL && (long)r0 * x->dim[k] >= TREE_ROWS_TALL) ||
            (r0 > TREE_RANK_TALL && (long)r1 * x->dim[k] >= TREE_ROWS_TALL))
            route = 2;
        if ((long)r0 * x->dim[k] > TREE_ROWS || (long)r1 * x->dim[k] > TREE_ROWS) return 0;
    }
    return route;
}

typedef struct {
    double sig[32];
    int info[4];
} bond_record;

/* from: the first core to factor; the cores before it are orthogonal, and the
 * train holds 2^-g_escale times the input. */
static double tree_round(attac_tt *x, const int *maxr, double tol, int tol_is_rel,
                         const double *rscale, const double *nscale, int from) {
    const int escale = g_escale;
    const int d = x->numDim;
    int *r = x->ttRank;
    const int *n = x->dim;
    ptt_tsqr_plan *pl = (ptt_tsqr_plan *)ptt_host_malloc(sizeof(ptt_tsqr_plan) * 2 * (size_t)d);
    ptt_tsqr_plan *pr = pl + d; /* right-to-left trees, by core */
    int *kept = (int *)ptt_host_malloc(sizeof(int) * (size_t)(d + 1)); /* largest rank left */
    for (int k = 0; k <= d; k++) kept[k] = (k > 0 && k < d && maxr[k] < r[k]) ? maxr[k] : r[k];
    for (int k = 0; k <= d; k++)
        if (kept[k] < 1) kept[k] = 1;
    /* one arena: the left-to-right trees' F and S per core, one right-to-left
     * tree's, two hand-down buffers each, the small matrices, the records */
    size_t fs = 0, rf = 0, rs = 0, w0 = 0, w1 = 0;
    size_t *off = (size_t *)ptt_host_malloc(sizeof(size_t) * 2 * (size_t)d);
    for (int i = 0; i < d; i++) {
        if (i < d - 1) {
            (void)ptt_hip_tsqr_plan(r[i + 1], (long)r[i] * n[i], &pl[i]);
            off[2 * i] = fs;
            off[2 * i + 1] = fs + (size_t)pl[i].fsize;
            if (i >= from) { /* before it: explicit Qs, level 0's blocks only */
                fs += (size_t)pl[i].fsize + (size_t)pl[i].ssize;
                if (pl[i].levels > 1 && (size_t)pl[i].lrows[1] > w1) w1 = (size_t)pl[i].lrows[1];
            }
        }
        if (i > 0) {
            (void)ptt_hip_tsqr_plan(r[i], (long)n[i] * kept[i + 1], &pr[i]);
            if ((size_t)pr[i].fsize > rf) rf = (size_t)pr[i].fsize;
            if ((size_t)pr[i].ssize > rs) rs = (size_t)pr[i].ssize;
            if (pr[i].levels > 1 && (size_t)pr[i].lrows[1] > w0) w0 = (size_t)pr[i].lrows[1];
        }
    }
    const size_t rec = sizeof(bond_record) / sizeof(double);
    double *ws = (double *)ptt_hip_scratch(
        PTT_WS_TREE, sizeof(double) * (fs + rf + rs + 64 * (w0 + w1) + 3 * 1024 +
                                       (rec + 1) * (size_t)d));
    double *F0 = ws + fs, *S0 = F0 + rf, *W0 = S0 + rs, *W1 = W0 + 64 * w0;
    double *R = W1 + 64 * w1, *X = R + 1024, *US = X + 1024, *records = US + 1024;
    int *rho = (int *)(records + rec * (size_t)d); /* device ranks, by bond */
    /* norm and exponent come back in one read */
    double *dss = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 24;
    ptt_hip_zero(dss, 2 * sizeof(double));
    for (int i = from; i < d - 1; i++) {
        const int c = r[i + 1];
        const long m = (long)r[i] * n[i], wcols = (long)n[i + 1] * r[i + 2];
        ptt_hip_tsqr_factor(&pl[i], x->coreList[i], 1, m, NULL, 0, ws + off[2 * i],
                            ws + off[2 * i + 1], R, (int *)(dss + 1));
        ptt_hip_dgemm('N', 'N', c, (int)wcols, c, rscale[i], R, c, x->coreList[i + 1], c, 0.0,
                      x->coreList[i + 1], c);
        if (i < 64) g_stats.ltr_cholqr_passes[i] = 0;
    }
    const int rl = r[d - 1];
    ptt_hip_sumsq(rl, n[d - 1] * r[d], x->coreList[d - 1], rl, dss);
    double back[2];
    ptt_hip_d2h(back, dss, sizeof back);
    double ss = back[0];
    memcpy(&g_escale, &back[1], sizeof(int));
    g_escale += escale;
    if (!(ss >= MAG_LO && ss <= MAG_HI)) ss = last_core_sumsq(x);
    const double nrm_s = sqrt(ss);
    const double abs_tol = tol_is_rel ? tol * nrm_s : ldexp(tol, -g_escale);
    const double delta = abs_tol / sqrt(d - 1.0);
    for (int i = d - 1; i > 0; i--) {
        const int c = r[i];
        const long wmax = (long)n[i] * kept[i + 1], m1 = (long)r[i - 1] * n[i - 1];
        const int *drho = (i == d - 1) ? NULL : rho + i + 1;
        double *sig = records + rec * (size_t)i;
        double *M = x->coreList[i], *A1 = x->coreList[i - 1];
        double *Y0 = (double *)ptt_hip_scratch(PTT_WS_TMP, sizeof(double) * (size_t)kept[i] * wmax);
        double *Y1 = (double *)ptt_hip_scratch(PTT_WS_TMP2, sizeof(double) * (size_t)m1 * kept[i]);
        ptt_hip_tsqr_factor(&pr[i], M, c, 1, drho, n[i], F0, S0, NULL, NULL);
        ptt_hip_tsqr_svd(&pr[i], M, c, 1, drho, n[i], F0, S0, delta, maxr[i], sig,
                         (int *)(sig + 32), rho + i, X, US, W0, Y0, nscale[i]);
        ptt_hip_tsqr_finish(&pr[i], M, drho, n[i], F0, S0, rho + i, W0, Y0, nscale[i], &pl[i - 1],
                            A1, i - 1 < from ? NULL : ws + off[2 * (i - 1)],
                            ws + off[2 * (i - 1) + 1], US, rho + i, W1, Y1, i == 1 ? nscale[0] : 1.0);
        ptt_host_swap_core_with_slot(x, i, (long)kept[i] * wmax, PTT_WS_TMP);
        ptt_host_swap_core_with_slot(x, i - 1, m1 * kept[i], PTT_WS_TMP2);
    }
    bond_record *h = (bond_record *)ptt_host_malloc(sizeof(bond_record) * (size_t)d);
    ptt_hip_d2h(h + 1, records + rec, sizeof(bond_record) * (size_t)(d - 1));
    for (int i = 1; i < d; i++) {
        const int k = h[i].info[1];
        if (i < 64) {
            const double *sv = h[i].sig;
            g_stats.numrank[i] = h[i].info[0];
            g_stats.svd_sweeps[i] = h[i].info[2];
            g_stats.rtl_cholqr_passes[i] = 0;
            g_stats.kappa_rtl[i] = sv[k - 1] > 0.0 ? sv[0] / sv[k - 1] : 0.0;
            for (int q = 0; q < 4; q++) {
                const int j = k - 1 + q;
                g_stats.sig[i][q] = j < 32 ? sv[j] : 0.0;
            }
            for (int q = 0; q < 16; q++) {
                const int j = k - 13 + q;
                g_spec[i][q] = (j >= 0 && j < 32) ? sv[j] : 0.0;
            }
            g_spec[i][16] = sv[0];
            g_spec[i][17] = k;
            g_spec[i][18] = r[i];
        }
        r[i] = k;
    }
    free(h); free(off); free(kept); free(pl);
    return nrm_s;
}

/* Shared driver: returns ||x||_n from the sweep (last core's Frobenius norm
 * in the scaled space). */
static double round_impl_g(attac_tt *x, const int *maxRank, double tol, int tol_is_rel,
                           int grid) {
    int d = x->numDim;
    memset(&g_stats, 0, sizeof g_stats);
    memset(g_spec, 0, sizeof g_spec);
    g_sketch_counts[0] = g_sketch_counts[1] = 0;
    g_stats.d = d;
    int *mr = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    memcpy(mr, maxRank, sizeof(int) * (d + 1)); /* maxRank may alias ttRank */
    double *inv = (double *)ptt_host_malloc(sizeof(double) * d);
    double *sq = (double *)ptt_host_malloc(sizeof(double) * d);
    double *qs = (double *)ptt_host_malloc(sizeof(double) * d);
    double *rs = (double *)ptt_host_malloc(sizeof(double) * d);
    fill_scales(x, inv, sq);
    if (!grid)
        for (int k = 0; k < d; k++) inv[k] = sq[k] = 1.0;
    for (int k = 0; k < d; k++) {
        qs[k] = 1.0;
        rs[k] = (k + 1 < d) ? inv[k + 1] : 1.0;
    }
    if (d >= 2) rs[0] *= inv[0];
    double nrm = 0.0;
    if (d >= 2) {
        g_escale = 0;
        double nrm_s;
        const int route = tree_route(x);
        q_factor *qf = NULL;
        if (route != 1) {
            size_t need = 0;
            qf = (q_factor *)calloc((size_t)d, sizeof *qf);
            if (!qf) {
                fprintf(stderr, "%s:Line %d %s::out of memory\n", __FILE__, __LINE__, __func__);
                exit(1);
            }
            for (int k = 0; k + 1 < d; k++)
                if (x->ttRank[k + 1] <= 128) need += (size_t)x->ttRank[k + 1] * x->ttRank[k + 1];
            double *t = need ? (double *)ptt_hip_scratch(PTT_WS_QFACT, sizeof(double) * need) : NULL;
            for (int k = 0; k + 1 < d; k++)
                if (x->ttRank[k + 1] <= 128) {
                    qf[k].t = t;
                    t += (size_t)x->ttRank[k + 1] * x->ttRank[k + 1];
                }
            g_qf = qf;
        }
        const int done = route == 1 ? 0 : ltr_sweep_until(x, qs, rs, route == 2);
        if (route == 1 || done < d - 1) {
            /* a train that changes over to the trees needs its Qs */
            for (int k = 0; k < done; k++)
                if (qf && qf[k].unformed)
                    apply_right(x, k, NULL, (long)x->ttRank[k] * x->dim[k], x->ttRank[k + 1],
                                qf[k].t, qf[k].alpha);
            nrm_s = tree_round(x, mr, tol, tol_is_rel, rs, sq, done);
        } else {
            /* norm in the scaled space: last core after the sweep (the train
             * holds 2^-g_escale times the input from here to the end) */
            const double ss = last_core_sumsq(x);
            nrm_s = sqrt(ss);
            const double abs_tol = tol_is_rel ? tol * nrm_s : ldexp(tol, -g_escale);
            rtl_sweep(x, mr, abs_tol, sq);
        }
        g_qf = NULL;
        free(qf);
        if (g_escale != 0) {
            /* core 0 carries the train's magnitude after the sweep */
            ptt_hip_scale(x->coreList[0], (long)x->ttRank[0] * x->dim[0] * x->ttRank[1],
                          ldexp(1.0, g_escale));
        }
        nrm = ldexp(nrm_s, g_escale);
        g_escale = 0;
    } else {
        /* one core: scale, nothing to orthogonalise or truncate, unscale */
        long cnt = (long)x->ttRank[0] * x->dim[0] * x->ttRank[1];
        double ss = 0.0;
        double *dss = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 24;
        ptt_hip_sumsq(1, (int)cnt, x->coreList[0], 1, dss);
        ptt_hip_d2h(&ss, dss, sizeof(double));
        nrm = sqrt(ss) * inv[0];
    }
    g_stats.norm = nrm;
    ptt_hip_sync();
    free(mr); free(inv); free(sq); free(qs); free(rs);
    return nrm;
}

static double round_impl(attac_tt *x, const int *maxRank, double tol, int tol_is_rel) {
    return round_impl_g(x, maxRank, tol, tol_is_rel, 1);
}

/* ---- public entry points ---- */

void paratt_truncate(paratt *x_ptt, double tol, int *maxRank) {
    round_impl(x_ptt->x, maxRank, tol, 0);
}

void paratt_amd_truncate_rel(paratt *x_ptt, double eps_rel, int *maxRank) {
    round_impl(x_ptt->x, maxRank, eps_rel, 1);
}

void paratt_amd_truncate_rel_sketch(paratt *x_ptt, double eps_rel, int *maxRank,
                                    const int *pred_rank) {
    attac_tt *x = x_ptt->x, *keep = NULL;
    const int d = x->numDim;
    /* No bond is large enough for a sketch of its prediction (ranks only fall on
     * the way): the plain rounding, decided before anything is queued. */
    int any = 0;
    for (int i = 1; pred_rank && i < d; i++)
        any = any || sketch_columns(pred_rank, i, x->ttRank[i],
                                    (long)x->dim[i] * x->ttRank[i + 1]) > 0;
    if (!any) {
        round_impl(x, maxRank, eps_rel, 1);
        return;
    }
    /* Refused predictions leave the plain rounding's result.  A train that it would
     * hand over to the trees (up to 32 columns and a core of more than one pass) is
     * kept until a step has been accepted. */
    int *mr = (int *)ptt_host_malloc(sizeof(int) * (size_t)(d + 1));
    memcpy(mr, maxRank, sizeof(int) * (size_t)(d + 1));
    if (tree_route(x)) {
        keep = alloc_tt(d, x->dim, x->ttRank);
        copy_rank_change_tt(keep, x);
    }
    g_pred = pred_rank;
    round_impl(x, mr, eps_rel, 1);
    g_pred = NULL;
    if (keep && g_sketch_counts[1] == 0 && g_sweep_multi) {
        const int tried = g_sketch_counts[0];
        copy_rank_change_tt(x, keep);
        round_impl(x, mr, eps_rel, 1);
        g_sketch_counts[0] = tried;
    }
    if (keep) free_tt(keep);
    free(mr);
}

void pattacTruncate(MPI_Comm comm, const int d, int *distrib_dim_mat, int *rx, double **x,
                    const int *maxr, const double abs_tol, const double rel_tol, const char ortho,
                    tsqr_tree *qrTree, int *int_wrk, double **flt_wrk_ptr, int *flt_sz_ptr) {
    (void)comm; (void)rel_tol; (void)qrTree; (void)int_wrk; (void)flt_wrk_ptr; (void)flt_sz_ptr;
    if (ortho != 'R') {
        fprintf(stderr, "%s:Line %d %s::Not known orthogonalization side\n", __FILE__, __LINE__,
                __func__);
        exit(1);
    }
    attac_tt view;
    ptt_host_view(&view, d, distrib_dim_mat, rx, x);
    round_impl(&view, maxr, abs_tol, 0);
    ptt_host_view_release(&view, x);
}

/* After a left-to-right sweep alone: the last core carries the train's
 * magnitude, so it takes the exponent of any rescaling back. */
static void ltr_unscale_last(attac_tt *x) {
    int d = x->numDim;
    if (g_escale != 0)
        ptt_hip_scale(x->coreList[d - 1], (long)x->ttRank[d - 1] * x->dim[d - 1] * x->ttRank[d],
                      ldexp(1.0, g_escale));
    g_escale = 0;
}

void pattacLOrthogonalization(MPI_Comm comm, int d, int *distrib_dim_mat, int *rx, double **x,
                              tsqr_tree *qrTree, int *int_wrk) {
    (void)comm; (void)qrTree; (void)int_wrk;
    attac_tt view;
    ptt_host_view(&view, d, distrib_dim_mat, rx, x);
    double *qs = (double *)ptt_host_malloc(sizeof(double) * d);
    double *rs = (double *)ptt_host_malloc(sizeof(double) * d);
    for (int k = 0; k < d; k++) { qs[k] = 1.0; rs[k] = 1.0; }
    g_escale = 0;
    if (d >= 2) ltr_sweep(&view, qs, rs);
    ltr_unscale_last(&view);
    ptt_hip_sync();
    ptt_host_view_release(&view, x);
    free(qs); free(rs);
}

void pattacLTruncate(MPI_Comm comm, const int d, int *distrib_dim_mat, int *rx, double **x,
                     const int *maxr, const double abs_tol, tsqr_tree *qrTree, int *int_wrk,
                     double **flt_wrk_ptr, int *flt_sz_ptr) {
    (void)comm; (void)qrTree; (void)int_wrk; (void)flt_wrk_ptr; (void)flt_sz_ptr;
    attac_tt view;
    ptt_host_view(&view, d, distrib_dim_mat, rx, x);
    double *ones = (double *)ptt_host_malloc(sizeof(double) * d);
    for (int k = 0; k < d; k++) ones[k] = 1.0;
    int *mr = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    memcpy(mr, maxr, sizeof(int) * (d + 1));
    if (d >= 2) {
        /* the input is left-orthogonal: its last core carries the magnitude */
        g_escale = 0;
        (void)last_core_sumsq(&view);
        rtl_sweep(&view, mr, ldexp(abs_tol, -g_escale), ones);
        if (g_escale != 0)
            ptt_hip_scale(view.coreList[0], (long)view.ttRank[0] * view.dim[0] * view.ttRank[1],
                          ldexp(1.0, g_escale));
        g_escale = 0;
    }
    ptt_hip_sync();
    ptt_host_view_release(&view, x);
    free(ones); free(mr);
}

/* ---- serial attac entry points (attac.h) ---- */

static void serial_view(attac_tt *view, int d, const int *n, int *r, double **x) {
    ptt_host_view(view, d, (int *)n, r, x);
}

void attacLOrthogonalization(const int d, const int *n, const int *rx, double **x,
                             double *work) {
    (void)work;
    for (int i = 0; i + 1 < d; i++)
        if ((long)rx[i] * n[i] < rx[i + 1]) {
            fprintf(stderr, "attacLOrthogonalization: rx[%d]*n[%d] = %ld < rx[%d] = %d\n", i, i,
                    (long)rx[i] * n[i], i + 1, rx[i + 1]);
            exit(1);
        }
    int *r = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    memcpy(r, rx, sizeof(int) * (d + 1));
    attac_tt view;
    serial_view(&view, d, n, r, x);
    double *ones = (double *)ptt_host_malloc(sizeof(double) * d);
    for (int k = 0; k < d; k++) ones[k] = 1.0;
    g_escale = 0;
    if (d >= 2) ltr_sweep(&view, ones, ones);
    ltr_unscale_last(&view);
    ptt_hip_sync();
    free(ones); free(r);
}

double attacNorm(const int d, const int *n, const int *rx, double **x, double *work) {
    (void)work;
    int *r = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    memcpy(r, rx, sizeof(int) * (d + 1));
    attac_tt view;
    serial_view(&view, d, n, r, x);
    const double v = attac_tt_norm(&view);
    ptt_hip_sync();
    free(r);
    return v;
}

void attacLTruncate(const int d, const int *n, int *rx, double **x, const int *maxr,
                    const double abs_tol, double *work) {
    (void)work;
    pattacLTruncate(0, d, (int *)n, rx, x, maxr, abs_tol, NULL, NULL, NULL, NULL);
}

void attacTruncate(const int d, const int *n, int *rx, double **x, const int *maxr,
                   const double abs_tol, const char ortho, double *work) {
    (void)work;
    if (ortho != 'R') {
        fprintf(stderr, "%s:Line %d %s::Not known orthogonalization side\n", __FILE__, __LINE__,
                __func__);
        exit(1);
    }
    attac_tt view;
    serial_view(&view, d, n, rx, x);
    round_impl_g(&view, maxr, abs_tol, 0, 0);
}

double paratt_norm(paratt *x_ptt) {
    attac_tt *x = x_ptt->x;
    int d = x->numDim;
    double *inv = (double *)ptt_host_malloc(sizeof(double) * d);
    double *sq = (double *)ptt_host_malloc(sizeof(double) * d);
    double *qs = (double *)ptt_host_malloc(sizeof(double) * d);
    double *rs = (double *)ptt_host_malloc(sizeof(double) * d);
    fill_scales(x, inv, sq);
    for (int k = 0; k < d; k++) {
        qs[k] = sq[k];                       /* leaves core k = sqrt(n_k) * Q_k */
        rs[k] = (k + 1 < d) ? inv[k + 1] : 1.0;
    }
    if (d >= 2) rs[0] *= inv[0];
    double *dss = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 24;
    double ss = 0.0;
    int ex = 0;
    if (d >= 2) {
        g_escale = 0;
        ltr_sweep(x, qs, rs);
        ss = last_core_sumsq(x);
        ex = g_escale;
        g_escale = 0;
        int rl = x->ttRank[d - 1];
        /* reference leaves the last core unscaled by sqrt(n_{d-1}) */
        ptt_hip_scale(x->coreList[d - 1], (long)rl * x->dim[d - 1], ldexp(sq[d - 1], ex));
    } else {
        long cnt = (long)x->ttRank[0] * x->dim[0] * x->ttRank[1];
        ptt_hip_sumsq(1, (int)cnt, x->coreList[0], 1, dss);
        ptt_hip_d2h(&ss, dss, sizeof(double));
        ss *= inv[0] * inv[0];
    }
    ptt_hip_sync();
    free(inv); free(sq); free(qs); free(rs);
    return ldexp(sqrt(ss), ex);
}

void attac_tt_truncate(attac_tt *x_tt, double tol, int *maxRank) {
    round_impl_g(x_tt, maxRank, tol, 0, 0);
}

double attac_tt_norm(attac_tt *x) {
    int d = x->numDim;
    double *dss = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 24;
    double ss = 0.0;
    if (d >= 2) {
        double *ones = (double *)ptt_host_malloc(sizeof(double) * d);
        for (int k = 0; k < d; k++) ones[k] = 1.0;
        g_escale = 0;
        ltr_sweep(x, ones, ones);
        free(ones);
        ss = last_core_sumsq(x);
        const int ex = g_escale;
        ltr_unscale_last(x);
        return ldexp(sqrt(ss), ex);
    }
    long cnt = (long)x->ttRank[0] * x->dim[0] * x->ttRank[1];
    ptt_hip_sumsq(1, (int)cnt, x->coreList[0], 1, dss);
    ptt_hip_d2h(&ss, dss, sizeof(double));
    return sqrt(ss);
}
