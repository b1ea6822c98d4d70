/* Launchers of the latent-to-PCM decoder's own kernels (pgpu_pcm.hip), for
 * host/phonon_audio.c. Everything here works on one pass of a request: all
 * of its positions at once, the positions before the pass taken from what
 * the pass before left behind.
 *
 * A "planes" buffer holds a convolution's input as the three exact bf16
 * terms of each value (hi + mid + lo): [3][channels / 8][stride][8] bf16, a
 * 16-byte slot per (term, 8 channels, position). Slot 16 + r is the pass's
 * position r; the 8 positions before the pass are slots 8 phase .. 8 phase
 * + 7, where the previous pass's producer put its last 8. phase alternates
 * from pass to pass, so a producer never writes what its pass's consumer
 * still reads. */
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
    int stride;   /* slots: 16 + the largest pass's positions */
} pgpu_planes;

/* Where a pass stands in its request. */
typedef struct {
    int phase; /* 0 or 1, alternating */
    int past;  /* 0: the request's first pass (what came before is zero) */
} pgpu_pass;

/* rows [positions][512] -> planes; positions >= 8. */
int pgpu_pcm_rows_to_planes(void *stream, const float *rows, int positions, const pgpu_planes *out,
                            pgpu_pass pass);

/* A convolution over planes: taps 7 (conv0: ncols = cout, ELU of the result
 * into `planes`) or taps 2 (a transposed convolution: ncols = stride * cout
 * columns k * cout + o per position, fp32 into `rows` [positions][ncols]).
 * in->channels is a multiple of 128, ncols and cout of 64; fragments as in
 * pgpu_conv_layer. positions >= 8. */
typedef struct {
    int taps, ncols, cout;
    const uint16_t *fragments;
    const float *bias;
} pgpu_plane_conv;
int pgpu_pcm_conv(void *stream, const pgpu_plane_conv *conv, const pgpu_planes *in, int positions,
                  pgpu_pass pass, float *rows, const pgpu_planes *planes, int *status);

/* A residual pair over x [positions][channels], channels 256, 128 or 64:
 * v = x + conv1(ELU(conv3(ELU(x)))). channels 256 and 128: ELU(v) into
 * `planes`. channels 64: the output convolution (3 taps, 64 -> 1) of ELU(v)
 * into pcm [positions]. history [2][4][channels] holds x's rows before the
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
