/* Launchers of the latent-to-PCM decoder's own kernels (pgpu_pcm.hip), for
 * host/phonon_audio.c. Everything here works on one pass of a request: all
 * of its positions at once, the positions before the pass taken from what
 * the pass before left behind.
 *
 * A "planes" buffer holds a convolution's input as the three exact bf16
 * terms of each value (hi + mid + lo): [3][channels / 8][stride][8] bf16, a
 * 16-byte slot per (term, 8 channels, position). Slot 8 + r is position r of
 * the pass, so that the 8 positions before it are slots 0 .. 7. */
#ifndef PGPU_PCM_H
#define PGPU_PCM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct {
    uint16_t *data;
    int channels; /* a multiple of 32 */
    int stride;   /* slots: 8 + the largest pass's positions */
} pgpu_planes;

/* Where a pass stands in its request. */
typedef struct {
    int phase; /* 0 or 1, alternating: which half of a residual pair's history */
    int past;  /* 0: the request's first pass (what came before is zero) */
} pgpu_pass;

/* What a request keeps of its convolutions' inputs between passes (the planes
 * themselves are only borrowed for a call): the last 8 positions of each,
 * [PGPU_KEPT_SLOTS] slots. */
enum { PGPU_KEPT_PLANES = 4, PGPU_KEPT_SLOTS = 8 * 3 * (512 + 512 + 256 + 128) / 8 };
typedef struct {
    pgpu_planes in[PGPU_KEPT_PLANES]; /* channels 512, 512, 256, 128 */
    int positions[PGPU_KEPT_PLANES];  /* of the pass */
    uint16_t *kept;
} pgpu_kept;

/* The first launch of a pass: pgpu_mimi_input (pgpu_audio.hip), whose
 * `latents` may be pinned host memory and whose `previous` is taken as zero
 * when past is 0, and, when it is 1 and keep given, the kept positions put
 * back before the pass's own. */
int pgpu_pcm_input(void *stream, const float *latents, int frames, const float *projection,
                   const float *upsample, float *previous, int past, const pgpu_kept *keep,
                   float *hidden, int *status);

/* The last one: the pass's last positions kept, and *seen = *status (seen:
 * pinned host memory); then the wait for an event recorded after it. */
int pgpu_pcm_keep(void *stream, const pgpu_kept *keep, const int *status, int *seen);
int pgpu_pcm_wait(void *event);

/* LayerNorm of rows [positions][512] -> planes. */
int pgpu_pcm_layer_norm(void *stream, const float *rows, const float *weight, const float *bias,
                        float epsilon, int positions, const pgpu_planes *out, int *status);

/* A product over planes, and what becomes of it. in->channels is a multiple
 * of 128 (512 for a projection), ncols of 64; fragments as in pgpu_conv_layer (a projection's
 * pgpu_matrix values are the same records); positions >= 8.
 *   ROWS   a transposed convolution: taps 2, ncols = stride * cout columns
 *          k * cout + o, + bias, fp32 into rows [positions][ncols]
 *   ELU    conv0: taps 7, + bias, ELU, into planes
 *   GELU   a projection (taps 1), GELU, into planes
 *   GATED  a projection to 512 columns: rows += gate * product, and, if
 *          planes.data is set, the sum into planes too
 *   QKV    the in-projection (1536 columns): RoPE of q and k at positions
 *          first + r, q into rows [positions][512], k and v into their ring
 *          slots (first + r) % ring */
enum { PGPU_PLANE_ROWS, PGPU_PLANE_ELU, PGPU_PLANE_GELU, PGPU_PLANE_GATED, PGPU_PLANE_QKV };
typedef struct {
    int epilogue, ncols, cout;
    const uint16_t *fragments;
    const float *bias; /* ROWS, ELU: [cout] */
    const float *gate; /* GATED: [512] */
    float *rows;
    pgpu_planes planes;
    const float *rope; /* QKV: [rope_positions][32] (cos, sin) */
    long long first, rope_positions;
    float *ring_k, *ring_v;
    int ring;
} pgpu_plane_product;
int pgpu_pcm_product(void *stream, const pgpu_plane_product *product, const pgpu_planes *in,
                     int positions, pgpu_pass pass, int *status);

/* pgpu_mimi_attention with q as QKV leaves it and its rows into planes. */
int pgpu_pcm_attention(void *stream, const float *q, int rows, long long first,
                       const float *ring_k, const float *ring_v, int ring, int context,
                       const pgpu_planes *out, int *status);

/* A residual pair over x [positions][channels], channels 256, 128 or 64:
 * v = x + conv1(ELU(conv3(ELU(x)))). channels 256 and 128: ELU(v) into
 * `planes`. channels 64: the output convolution (3 taps, 64 -> 1) of ELU(v)
 * into pcm [positions] (device or pinned host memory). history [2][4][channels] holds x's rows before the
 * pass (by phase) and receives its last four. positions >= 8. */
typedef struct {
    const uint16_t *conv3, *conv1, *last; /* fragments; last: channels 64 only */
    const float *bias3, *bias1, *bias_last;
} pgpu_residual_weights;
int pgpu_pcm_residual(void *stream, const pgpu_residual_weights *w, int channels, const float *x,
                      int positions, pgpu_pass pass, float *history, const pgpu_planes *planes,
                      float *pcm, int *status);

#ifdef __cplusplus
}
#endif
#endif
