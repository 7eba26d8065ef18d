/* mds_stage.h -- host side of the state's way back: staged values into the
 * caller's array (mds_stage.c). */
#ifndef MDS_STAGE_H
#define MDS_STAGE_H
#ifdef __cplusplus
extern "C" {
#endif
/* d[0..n) = s[0..n), widened (fp32) or copied; large arrays by several threads */
void mds_stage_out(double *d, const void *s, int fp32, long long n);
#ifdef __cplusplus
}
#endif
#endif
