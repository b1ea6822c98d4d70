/* The device calls of host/phonon_audio.c on host memory, for CPU tests of what
 * that file allocates: kernels do nothing, `waiting` calls meet at a barrier in
 * the wait for their last kernel (so that many are in flight at once), and the
 * allocations are counted and can be made to fail. */
#include "../speech-mac_amd/csrc/pgpu_pcm.h"
#include "../speech-mac_amd/host/ph_internal.h"
#include "phonon_pack.h"

#include <pthread.h>
#include <stdlib.h>
#include <string.h>

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t met = PTHREAD_COND_INITIALIZER;
static int waiting, arrived, round_no, failing, made, released;
static size_t held;

void stub_wait_for(int calls) { waiting = calls; }
void stub_fail(int fail) { failing = fail; }
int stub_made(void) { return made; }
int stub_released(void) { return released; }
size_t stub_held(void) { return held; }

static void *take(size_t bytes) {
    pthread_mutex_lock(&lock);
    size_t *p = failing ? NULL : calloc(1, bytes + 256);
    if (p) {
        made++;
        held += bytes;
        p[0] = bytes;
    }
    pthread_mutex_unlock(&lock);
    return p ? (char *)p + 256 : NULL;
}

static void give(void *at) {
    if (!at)
        return;
    size_t *p = (size_t *)((char *)at - 256);
    pthread_mutex_lock(&lock);
    released++;
    held -= p[0];
    pthread_mutex_unlock(&lock);
    free(p);
}

void *pgpu_malloc(size_t bytes) { return take(bytes); }
void pgpu_free(void *p) { give(p); }
void *pgpu_host_malloc(size_t bytes) { return take(bytes); }
void pgpu_host_free(void *p) { give(p); }
int pgpu_event_create(void **event) { return (*event = take(1)) != NULL; }
void pgpu_event_destroy(void *event) { give(event); }
int pgpu_event_record(void *event, void *stream) { return event && stream; }
int pgpu_stream_create(void **stream) { return (*stream = take(1)) != NULL; }
void pgpu_stream_destroy(void *stream) { give(stream); }
int pgpu_stream_sync(void *stream) { return (void)stream, 1; }
int pgpu_device_init(void) { return 1; }
void pgpu_record_error(const char *message) { (void)message; }
const char *pgpu_last_error(void) { return ""; }
int pgpu_memset(void *stream, void *dst, int value, size_t bytes) {
    return (void)stream, memset(dst, value, bytes), 1;
}
int pgpu_copy_h2d(void *stream, void *dst, const void *src, size_t bytes) {
    return (void)stream, memcpy(dst, src, bytes), 1;
}
int pgpu_copy_d2h(void *stream, void *dst, const void *src, size_t bytes) {
    return (void)stream, memcpy(dst, src, bytes), 1;
}

int pgpu_pcm_input(void *stream, const float *latents, int frames, const float *projection,
                   const float *upsample, float *previous, int past, const pgpu_kept *keep,
                   float *hidden, int *status) {
    (void)stream, (void)latents, (void)frames, (void)projection, (void)upsample, (void)previous;
    (void)past, (void)keep, (void)hidden, (void)status;
    return 1;
}

int pgpu_pcm_layer_norm(void *stream, const float *rows, const float *weight, const float *bias,
                        float epsilon, int positions, const pgpu_planes *out, int *status) {
    (void)stream, (void)rows, (void)weight, (void)bias, (void)epsilon, (void)status;
    return out->stride >= 8 + positions;
}

int pgpu_pcm_product(void *stream, const pgpu_plane_product *product, const pgpu_planes *in,
                     int positions, pgpu_pass pass, int *status) {
    (void)stream, (void)product, (void)pass, (void)status;
    return in->stride >= 8 + positions;
}

int pgpu_pcm_attention(void *stream, const float *q, int rows, long long first,
                       const float *ring_k, const float *ring_v, int ring, int context,
                       const pgpu_planes *out, int *status) {
    (void)stream, (void)q, (void)first, (void)ring_k, (void)ring_v, (void)ring, (void)context;
    (void)status;
    return out->stride >= 8 + rows;
}

int pgpu_pcm_residual(void *stream, const pgpu_residual_weights *w, int channels, const float *x,
                      int positions, pgpu_pass pass, float *history, const pgpu_planes *planes,
                      float *pcm, int *status) {
    (void)stream, (void)w, (void)channels, (void)x, (void)pass, (void)history, (void)status;
    if (pcm)
        memset(pcm, 0, (size_t)positions * sizeof(float));
    return !planes || planes->stride >= 8 + positions;
}

int pgpu_pcm_keep(void *stream, const pgpu_kept *keep, const int *status, int *seen) {
    (void)stream, (void)keep, (void)status;
    *seen = 0;
    return 1;
}

int pgpu_pcm_wait(void *event) {
    (void)event;
    pthread_mutex_lock(&lock);
    if (waiting > 1) {
        const int mine = round_no;
        if (++arrived == waiting) {
            arrived = 0;
            round_no++;
            pthread_cond_broadcast(&met);
        }
        while (round_no == mine)
            pthread_cond_wait(&met, &lock);
    }
    pthread_mutex_unlock(&lock);
    return 1;
}

/* Not called: phonon_audio.c's single convolutions and pack loader. */
int pgpu_elu(void *stream, const float *x, float *y, size_t count) {
    return (void)stream, (void)x, (void)y, (void)count, 0;
}

int pgpu_conv_rows(void *stream, const pgpu_conv_layer *layer, const float *x, int positions,
                   const float *history, float *history_out, const float *residual, int elu,
                   float *y, int *status) {
    (void)stream, (void)layer, (void)x, (void)positions, (void)history, (void)history_out;
    return (void)residual, (void)elu, (void)y, (void)status, 0;
}

int pgpu_upsample_frame(void *stream, const float *kernel, const float *input,
                        const float *previous, int channels, int stride, float *output,
                        int *status) {
    (void)stream, (void)kernel, (void)input, (void)previous, (void)channels, (void)stride;
    return (void)output, (void)status, 0;
}

int phonon_pack_tensor(const PhononPack *pack, const char *name, PhononTensorView *view) {
    return (void)pack, (void)name, (void)view, 0;
}
