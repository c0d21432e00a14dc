/* sep_host.h -- host-side C parts of libsep: the double-double Cholesky that
 * decides the ortho cutoff (the reference's SVD is Intel MKL's,
 * filter/ortho.c:32) and helpers shared by the C-ABI layer.  Internal to the
 * library. */
#ifndef SEP_HOST_H
#define SEP_HOST_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Upper Cholesky of G = hi + lo (double-double, n x n row-major) + shift*I,
 * carried out in double-double; R (rounded to double) gets the factor.
 * Returns 0 or k+1 for a non-positive pivot k. */
int sep_la_chol_dd(long n, const double *hi, const double *lo, double shift, double *R);

/* Ring depths (Newton vectors of one block) of nd filters that run together: nc
 * Newton vectors in all, ms targets and per_k bytes a vector of each, at most
 * `most`.  Where the rings exceed `total` bytes, the deepest are halved first. */
void sep_ring_plan(int nd, const long *nc, const long *ms, const double *per_k, long most,
                   double total, long *K);
/* The next depth where the memory is short: half of k, in whole sixteens. */
long sep_ring_halve(long k);

/* Up to eight threads (the caller's among them, no more than the CPUs it may
 * run on) that copy large host blocks together: first touches of a fresh
 * destination dominate such copies and run in parallel.  One download at a time:
 * wake, any number of runs, rest; the threads sleep outside of it.  NULL, where
 * memory is short, is a valid team of the caller alone. */
typedef struct sep_copy_team sep_copy_team;
sep_copy_team *sep_copy_team_open(void);
void sep_copy_team_wake(sep_copy_team *t);
void sep_copy_team_run(sep_copy_team *t, void *dst, const void *src, size_t n);
void sep_copy_team_rest(sep_copy_team *t);
void sep_copy_team_close(sep_copy_team *t);

#ifdef __cplusplus
}
#endif
#endif
