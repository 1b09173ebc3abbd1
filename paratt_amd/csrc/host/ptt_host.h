/* ptt_host.h -- internal helpers shared by the C host files. */
#ifndef PARATT_AMD_PTT_HOST_H
#define PARATT_AMD_PTT_HOST_H

#include "paratt.h"

/* Make core k's buffer the TMP scratch buffer (which holds the result of an
 * out-of-place kernel) and give the old buffer to the scratch slot.  For a
 * borrowed view (coreMem == NULL) the result is copied back instead, so the
 * caller's pointers never change (`count` doubles of result). */
void ptt_host_swap_core_with_tmp(attac_tt *x, int k, long count);
void ptt_host_swap_core_with_slot(attac_tt *x, int k, long count, int slot); /* another slot */
/* Roundings keep every bond's whole spectrum, also below the resolution of
 * FP64 (the rank predictor's features and training data): on = 1. */
void ptt_host_whole_spectra(int on);
/* Set the diagonal of an m x m device matrix to alpha. */
void ptt_host_set_diag(double *A, int m, double alpha);
/* Wrap raw (d, n, r, cores) arrays of the pattac* API as a borrowed TT. */
void ptt_host_view(attac_tt *view, int d, int *n, int *r, double **x);
void ptt_host_view_release(attac_tt *view, double **x);
/* Ensure core k of x can hold count[k] doubles, for every core (contents of
 * cores that grow are not preserved). */
void ptt_host_reserve_train(attac_tt *x, const long *count);
/* Upload a small host coefficient vector to the COEF scratch slot. */
double *ptt_host_coef(const double *host, long count);
void ptt_host_fatal(const char *fn, const char *msg);
/* Host allocations that print and exit on failure, like the rest of the
 * library's fatal paths. */
#include <stddef.h>
void *ptt_host_malloc(size_t bytes);
void *ptt_host_calloc(size_t count, size_t size);
void *ptt_host_realloc(void *p, size_t bytes);

#endif
