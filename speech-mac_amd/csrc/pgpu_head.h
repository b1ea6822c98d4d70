/* Launcher of pgpu_head.hip that only host/phonon_flow_head.c calls. */
#ifndef PGPU_HEAD_H
#define PGPU_HEAD_H

#include "phonon_gpu.h"

#ifdef __cplusplus
extern "C" {
#endif

/* pgpu_head_mlp_in beside an adaLN projection that a later launch reads:
 * next_mod [streams][ld_mod] = next_ada . silu + next_bias. */
int pgpu_head_mlp_in_beside(void *stream, const pgpu_matrix *w, const float *x, int streams,
                            const float *norm_w, const float *norm_b, float eps, const float *mod,
                            int ld_mod, const float *bias, uint16_t *out_split,
                            const pgpu_matrix *next_ada, const uint16_t *silu_split,
                            const float *next_bias, float *next_mod, int *status);

#ifdef __cplusplus
}
#endif
#endif
