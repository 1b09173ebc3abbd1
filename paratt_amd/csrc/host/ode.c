/*
 * ode.c -- step-truncation explicit Euler (paratt_ode.c:13-37) over the
 * GPU-resident primitives.  The vector field is the caller's host C code.
 */
#include "paratt.h"
#include "paratt_ode.h"
#include "ptt_host.h"

/* paratt_ode.c:26-37: f_new = T2(f_old + dt*T1(F(f_old))), caps = current ranks. */
void pattac_exp_euler_st(paratt *f_old, paratt *f_new, paratt *work,
                         void (*vecField)(paratt *, paratt *, int, ...), double dt, double eps_1,
                         double eps_2) {
    vecField(f_old, work, 0);
    paratt_truncate(work, eps_1, work->x->ttRank);
    attac_tt_axpby(1.0, f_old->x, dt, work->x, f_new->x);
    paratt_truncate(f_new, eps_2, f_new->x->ttRank);
}

/* paratt_ode.c:13-24: both truncations go through attac_tt_truncate, as in
 * the reference (plain Frobenius norm, absolute tolerance; the reference's
 * serial version has its SVD calls commented out, this one is the GPU
 * rounding without the grid scaling). */
void attac_exp_euler_st(attac_tt *f_old, attac_tt *f_new, attac_tt *work,
                        void (*vecField)(attac_tt *, attac_tt *, int, ...), double dt,
                        double eps_1, double eps_2) {
    vecField(f_old, work, 0);
    attac_tt_truncate(work, eps_1, work->ttRank);
    attac_tt_axpby(1.0, f_old, dt, work, f_new);
    attac_tt_truncate(f_new, eps_2, f_new->ttRank);
}

/* ------------------------------------------------------------------ */
/* Reaction-Burgers field and step-truncation RK4 (project composite;  */
/* the reference ships only explicit Euler).                           */
/* ------------------------------------------------------------------ */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "paratt_amd.h"
#include "ptt_hip.h"

static paratt *ptt_clone(paratt *s) {
    paratt *p = alloc_ptt(s->numDim, s->dim, s->x->ttRank);
    copy_rank_change_tt(p->x, s->x);
    return p;
}

static paratt *ptt_axpby_new(double a, paratt *x, double b, paratt *y) {
    int d = x->numDim;
    int *rz = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++)
        rz[k] = (k == 0 || k == d) ? 1 : x->x->ttRank[k] + y->x->ttRank[k];
    paratt *z = alloc_ptt(d, x->dim, rz);
    attac_tt_axpby(a, x->x, b, y->x, z->x);
    free(rz);
    return z;
}

/* ---- learned rank prediction for the step truncations -------------------
 * Every truncation site of the composite (role) keeps the spectrum record of
 * its last rounding.  In learned mode the rank-predictor network maps, per
 * bond, that record to a predicted rank, which sizes the sketched step of
 * paratt_amd_truncate_rel_sketch; in logging mode the (features, new rank)
 * pairs of plain roundings are collected as training data.
 * Features (18, FP32): log10(sigma_{rho-13+q}/sigma_0)/16 for q = 0..15
 * from the previous rounding of this site (-20/16 where absent), bond index
 * i/(d-1), and the previous kept rank rho/64.  Target: the new rank / 64. */
enum { ROLE_V, ROLE_HD, ROLE_F, ROLE_U2, ROLE_U3, ROLE_U4, ROLE_S, ROLE_UN, NROLES };
#define LN_FEAT 18
#define LN_SPEC 20
static struct {
    int valid, d;
    double spec[64][LN_SPEC];
} g_hist[NROLES];
static struct {
    int mode;
    float *dP;  /* device parameters */
    int nparam;
    int log_on, nlog, caplog;
    float *logX, *logY;
    long n_pred, n_att, n_acc;
} g_learn;

static void make_features(const double *spec, int i, int d, float *f) {
    const double s0 = spec[16];
    for (int q = 0; q < 16; q++) {
        double v = (spec[q] > 0.0 && s0 > 0.0) ? log10(spec[q] / s0) : -20.0;
        if (v < -20.0) v = -20.0;
        f[q] = (float)(v / 16.0);
    }
    f[16] = (float)((double)i / (double)(d > 1 ? d - 1 : 1));
    f[17] = (float)(spec[17] / 64.0);
}

void paratt_amd_learned_set_params(const float *P, int nparam) {
    if (nparam != ptt_hip_mlp_nparam()) {
        fprintf(stderr, "paratt_amd: rank predictor expects %d parameters, got %d\n",
                ptt_hip_mlp_nparam(), nparam);
        exit(1);
    }
    if (!g_learn.dP) g_learn.dP = (float *)ptt_hip_malloc(sizeof(float) * (size_t)nparam);
    ptt_hip_h2d(g_learn.dP, P, sizeof(float) * (size_t)nparam);
    g_learn.nparam = nparam;
}

void paratt_amd_learned_mode(int on) {
    if (on == 1 && !g_learn.dP) {
        fprintf(stderr, "paratt_amd: learned mode needs paratt_amd_learned_set_params first\n");
        exit(1);
    }
    g_learn.mode = on;
}

void paratt_amd_learned_reset_history(void) { memset(g_hist, 0, sizeof g_hist); }

void paratt_amd_learned_log(int on, int capacity) {
    g_learn.log_on = on;
    if (on && capacity > g_learn.caplog) {
        g_learn.logX = (float *)ptt_host_realloc(g_learn.logX, sizeof(float) * LN_FEAT * (size_t)capacity);
        g_learn.logY = (float *)ptt_host_realloc(g_learn.logY, sizeof(float) * (size_t)capacity);
        g_learn.caplog = capacity;
    }
    if (on) g_learn.nlog = 0;
}

int paratt_amd_learned_log_fetch(float *X, float *Y, int max) {
    int n = g_learn.nlog < max ? g_learn.nlog : max;
    memcpy(X, g_learn.logX, sizeof(float) * LN_FEAT * (size_t)n);
    memcpy(Y, g_learn.logY, sizeof(float) * (size_t)n);
    return n;
}

void paratt_amd_learned_counts(long *out) {
    out[0] = g_learn.n_pred;
    out[1] = g_learn.n_att;
    out[2] = g_learn.n_acc;
}

static void round_rel_cap_role(paratt *x, double eps, int cap, int role) {
    int d = x->numDim;
    int *mr = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++) mr[k] = (k == 0 || k == d) ? 1 : cap;
    ptt_host_whole_spectra(g_learn.mode != 0 || g_learn.log_on);
    const int have = (role >= 0 && g_hist[role].valid && g_hist[role].d == d && d <= 64);
    float *feat = NULL;
    if (have && (g_learn.mode == 1 || g_learn.log_on)) {
        feat = (float *)ptt_host_malloc(sizeof(float) * LN_FEAT * (size_t)d);
        for (int i = 1; i < d; i++) make_features(g_hist[role].spec[i], i, d, feat + LN_FEAT * (i - 1));
    }
    if (g_learn.mode == 2 && have) {
        /* heuristic baseline: the previous rank as the prediction */
        int *pred = (int *)ptt_host_calloc((size_t)d + 1, sizeof(int));
        for (int i = 1; i < d; i++) pred[i] = (int)g_hist[role].spec[i][17];
        paratt_amd_truncate_rel_sketch(x, eps, mr, pred);
        int c2[2];
        paratt_amd_last_sketch_counts(c2);
        g_learn.n_pred++;
        g_learn.n_att += c2[0];
        g_learn.n_acc += c2[1];
        free(pred);
    } else if (g_learn.mode == 1 && feat) {
        /* one forward launch for all bonds */
        int ns = d - 1;
        float *dX = (float *)ptt_hip_scratch(PTT_WS_COEF, sizeof(float) * (LN_FEAT + 1) * (size_t)ns + 64);
        float *dO = dX + LN_FEAT * ns;
        ptt_hip_h2d_queued(dX, feat, sizeof(float) * LN_FEAT * (size_t)ns);
        ptt_hip_mlp_forward(ns, dX, g_learn.dP, dO);
        float *out = (float *)ptt_host_malloc(sizeof(float) * (size_t)ns);
        ptt_hip_d2h(out, dO, sizeof(float) * (size_t)ns);
        int *pred = (int *)ptt_host_calloc((size_t)d + 1, sizeof(int));
        for (int i = 1; i < d; i++) {
            long p = lrint(64.0 * out[i - 1]);
            pred[i] = p < 1 ? 1 : (p > 1024 ? 1024 : (int)p);
        }
        paratt_amd_truncate_rel_sketch(x, eps, mr, pred);
        int c2[2];
        paratt_amd_last_sketch_counts(c2);
        g_learn.n_pred++;
        g_learn.n_att += c2[0];
        g_learn.n_acc += c2[1];
        free(pred);
        free(out);
    } else {
        paratt_amd_truncate_rel(x, eps, mr);
    }
    ptt_host_whole_spectra(0);
    if (role >= 0) {
        double spec[64 * LN_SPEC];
        paratt_amd_last_round_spectra(spec);
        if (g_learn.log_on && feat) {
            for (int i = 1; i < d && g_learn.nlog < g_learn.caplog; i++) {
                memcpy(g_learn.logX + LN_FEAT * (size_t)g_learn.nlog, feat + LN_FEAT * (i - 1),
                       sizeof(float) * LN_FEAT);
                g_learn.logY[g_learn.nlog] = (float)(spec[i * LN_SPEC + 17] / 64.0);
                g_learn.nlog++;
            }
        }
        memcpy(g_hist[role].spec, spec, sizeof spec);
        g_hist[role].valid = 1;
        g_hist[role].d = d;
    }
    free(feat);
    free(mr);
}

static void round_rel_cap(paratt *x, double eps, int cap) { round_rel_cap_role(x, eps, cap, -1); }

void paratt_amd_mode_sum(paratt *u, const double *sten3, paratt *s) {
    int d = u->numDim;
    int *rs = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++) rs[k] = (k == 0 || k == d) ? 1 : 2 * u->x->ttRank[k];
    rank_change_tt(s->x, rs);
    ptt_hip_mode_sum_train(d, u->dim, u->x->ttRank, u->x->coreList, sten3, s->x->coreList);
    ptt_hip_sync();
    free(rs);
}

static struct {
    double nu, h, eps;
    int cap;
} g_rb = {0.01, 1.0, 1e-8, 64};

void paratt_amd_rxn_burgers_setup(double nu, double h, double eps, int cap) {
    g_rb.nu = nu;
    g_rb.h = h;
    g_rb.eps = eps;
    g_rb.cap = cap;
}

/* out = u .* T(1 - u - sum_i D1_i u) + nu * sum_i D2_i u  (vecField-compatible) */
void paratt_amd_rxn_burgers_field(paratt *u, paratt *out, int nargs, ...) {
    (void)nargs;
    int d = u->numDim;
    double h = g_rb.h;
    double d1[3] = {-0.5 / h, 0.0, 0.5 / h};
    double d2[3] = {1.0 / (h * h), -2.0 / (h * h), 1.0 / (h * h)};
    int *one = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++) one[k] = 1;
    paratt *ones = alloc_ptt(d, u->dim, one);
    for (int k = 0; k < d; k++) ptt_hip_fill(ones->x->coreList[k], u->dim[k], 1.0);
    paratt *s1 = alloc_ptt(d, u->dim, one);
    paratt *lap = alloc_ptt(d, u->dim, one);
    paratt_amd_mode_sum(u, d1, s1);
    paratt_amd_mode_sum(u, d2, lap);
    paratt *v0 = ptt_axpby_new(1.0, ones, -1.0, u);
    paratt *v = ptt_axpby_new(1.0, v0, -1.0, s1);
    round_rel_cap_role(v, g_rb.eps, g_rb.cap, ROLE_V);
    int *rh = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++) rh[k] = u->x->ttRank[k] * v->x->ttRank[k];
    paratt *hd = alloc_ptt(d, u->dim, rh);
    pattacHadamard(d, u->dim, u->x->ttRank, u->x->coreList, v->x->ttRank, v->x->coreList,
                   hd->x->ttRank, hd->x->coreList);
    round_rel_cap_role(hd, g_rb.eps, g_rb.cap, ROLE_HD);
    paratt *f = ptt_axpby_new(1.0, hd, g_rb.nu, lap);
    round_rel_cap_role(f, g_rb.eps, g_rb.cap, ROLE_F);
    copy_rank_change_tt(out->x, f->x);
    free_ptt(ones); free_ptt(s1); free_ptt(lap); free_ptt(v0); free_ptt(v); free_ptt(hd);
    free_ptt(f);
    free(one); free(rh);
}

/* Step-truncation RK4: stages and the final combination are rounded to eps
 * (relative) with the rank cap; vecField rounds its own output. */
void paratt_amd_rk4_st(paratt *f_old, paratt *f_new,
                       void (*vecField)(paratt *, paratt *, int, ...), double dt, double eps,
                       int cap) {
    int d = f_old->numDim;
    int *one = (int *)ptt_host_malloc(sizeof(int) * (d + 1));
    for (int k = 0; k <= d; k++) one[k] = 1;
    paratt *k1 = alloc_ptt(d, f_old->dim, one), *k2 = alloc_ptt(d, f_old->dim, one);
    paratt *k3 = alloc_ptt(d, f_old->dim, one), *k4 = alloc_ptt(d, f_old->dim, one);
    vecField(f_old, k1, 0);
    paratt *u2 = ptt_axpby_new(1.0, f_old, 0.5 * dt, k1);
    round_rel_cap_role(u2, eps, cap, ROLE_U2);
    vecField(u2, k2, 0);
    paratt *u3 = ptt_axpby_new(1.0, f_old, 0.5 * dt, k2);
    round_rel_cap_role(u3, eps, cap, ROLE_U3);
    vecField(u3, k3, 0);
    paratt *u4 = ptt_axpby_new(1.0, f_old, dt, k3);
    round_rel_cap_role(u4, eps, cap, ROLE_U4);
    vecField(u4, k4, 0);
    paratt *s12 = ptt_axpby_new(1.0, k1, 2.0, k2);
    paratt *s123 = ptt_axpby_new(1.0, s12, 2.0, k3);
    paratt *s = ptt_axpby_new(1.0, s123, 1.0, k4);
    round_rel_cap_role(s, eps, cap, ROLE_S);
    paratt *un = ptt_axpby_new(1.0, f_old, dt / 6.0, s);
    round_rel_cap_role(un, eps, cap, ROLE_UN);
    copy_rank_change_tt(f_new->x, un->x);
    free_ptt(k1); free_ptt(k2); free_ptt(k3); free_ptt(k4); free_ptt(u2); free_ptt(u3);
    free_ptt(u4); free_ptt(s12); free_ptt(s123); free_ptt(s); free_ptt(un);
    free(one);
}
