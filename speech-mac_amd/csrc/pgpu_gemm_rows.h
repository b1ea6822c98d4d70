/* Launcher of pgpu_gemm.hip that only host/phonon_q8.c calls. */
#ifndef PGPU_GEMM_ROWS_H
#define PGPU_GEMM_ROWS_H

#include "phonon_gpu.h"

#ifdef __cplusplus
extern "C" {
#endif

/* out[s][r] = sum_c rows[s][c] W[r][c] for fp32 rows [streams][W->columns] of
 * any K, 16-byte aligned: one launch, the bits of pgpu_split_rows followed by
 * pgpu_gemm_store. */
int pgpu_gemm_store_rows(void *stream, const pgpu_matrix *w, const float *rows, int streams,
                         float *out, int ld_out, int *status);

#ifdef __cplusplus
}
#endif
#endif
