/* Launchers of pgpu_prefill.hip that only host/phonon_flow_batch.c calls. */
#ifndef PGPU_PREFILL_H
#define PGPU_PREFILL_H

#include <stdint.h>

#include "phonon_gpu.h"

#ifdef __cplusplus
extern "C" {
#endif

/* pgpu_prefill_attention_mfma's contract for pairs whose runs have at most 16
 * positions each, with exact fp32 products and PGPU_SPLIT_F16_PAIR outputs: a
 * work-group per (run, head), its keys dealt to four waves. */
int pgpu_prefill_attention_short(void *stream, const float *q, const pgpu_paged_kv *kv, int layer,
                                 const int32_t *tables, int table_stride,
                                 const int32_t *positions, int streams, const int32_t *pairs,
                                 int pair_count, uint16_t *out_split, int *status);

#ifdef __cplusplus
}
#endif
#endif
