/*
 * mds_stage.c -- staged state values into the caller's array.
 *
 * The caller's array is usually fresh memory, whose pages are faulted in by
 * the first store: one thread writes it at some 5 GB/s, so large pieces are
 * shared out (a 256^3 FP32 state, 671 MB of doubles: 122 ms with one
 * thread and pageable copies, 15.5 ms with eight beside the copy of the next piece).
 */
#include <string.h>
#include "../common/mds_stage.h"

#define STAGE_PIECE (1LL << 14)     /* values a thread takes at a time */
#define STAGE_THREADS 8

void mds_stage_out(double *d, const void *s, int fp32, long long n)
{
  const long long pieces = (n + STAGE_PIECE - 1) / STAGE_PIECE;
#pragma omp parallel for schedule(static) num_threads(STAGE_THREADS) if (pieces >= 2 * STAGE_THREADS)
  for (long long k = 0; k < pieces; k++) {
    const long long a = k * STAGE_PIECE, m = n - a < STAGE_PIECE ? n - a : STAGE_PIECE;
    if (fp32) {
      const float *f = (const float *)s + a;
      double *o = d + a;
#pragma omp simd
      for (long long q = 0; q < m; q++) o[q] = f[q];
    } else {
      memcpy(d + a, (const double *)s + a, (size_t)m * sizeof(double));
    }
  }
}
