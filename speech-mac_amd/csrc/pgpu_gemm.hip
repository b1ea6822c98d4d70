// Single-phase projection kernels: one projection of B streams per launch,
// one task (pgpu_gemm.hpp) per 512-thread work-group. Used by the primitives
// of phonon_transformer.h / phonon_q8.h and by the batched step when it runs
// phase by phase; the one-launch step (pgpu_flow.hip) runs the same tasks.
#include "pgpu_gemm.hpp"
#include "pgpu_gemm_rows.h"
#include "phonon_gpu.h"

namespace pgpu {

template <int EPI, bool Q8>
__global__ __launch_bounds__(kTaskThreads) void k_gemm(GemmArgs a) {
    __shared__ f32x4 lds4[kTaskWaves * 64];
    gemm_split_task<EPI, Q8>(a, blockIdx.x, blockIdx.y, (uint16_t *)lds4, NoWait{});
}

template <int SRC, int EPI, bool Q8>
__global__ __launch_bounds__(kTaskThreads) void k_gemm_wide(GemmArgs a) {
    __shared__ uint4 bsh4[kTaskLds / 8];
    gemm_wide_task<SRC, EPI, Q8>(a, blockIdx.x, blockIdx.y, (uint16_t *)bsh4, NoWait{});
}

// gemm_split_task on fp32 rows (a.ln_x, [streams][k_cols]) and Q8 weights: a lane
// splits its 8 columns of each block itself, CH blocks of its wave's range
// requested at once (all of them up to K = 2048). Every row tile's work-group
// splits the rows again, which is less than the launch that would do it for them
// as long as the work-groups run at once: a 512 x 2048 product of one row is bound
// by its launches and load latencies (7.5 us with the rows split by a launch of
// their own, 5.2 with this).
template <int CH>
__global__ __launch_bounds__(kTaskThreads) void k_gemm_rows(GemmArgs a) {
    __shared__ f32x4 partial[kTaskWaves * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, tile = blockIdx.x, st = blockIdx.y;
    const int kbn = a.k_cols >> 5, per = (kbn + kTaskWaves - 1) / kTaskWaves;
    const int kb_begin = wave * per, kb_end = min(kbn, kb_begin + per);
    const int s = st * 16 + (lane & 15), row0 = tile * 16 + (lane >> 4) * 4;
    const bool live = s < a.streams;
    const float *row = a.ln_x + (size_t)(live ? s : 0) * a.k_cols + 8 * (lane >> 4);
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    bool bad = false;
    for (int kb0 = kb_begin; kb0 < kb_end; kb0 += CH) {
        WChunk<true, CH> w;
        load_weights(w, a, tile, kbn, lane, kb0, kb_end);
        float4 x[CH][2];
#pragma unroll
        for (int u = 0; u < CH; u++) {
            const float4 *src = (const float4 *)(row + min(kb0 + u, kb_end - 1) * 32);
            x[u][0] = src[0];
            x[u][1] = src[1];
        }
#pragma unroll
        for (int u = 0; u < CH; u++) {
            const float v[8] = {x[u][0].x, x[u][0].y, x[u][0].z, x[u][0].w,
                                x[u][1].x, x[u][1].y, x[u][1].z, x[u][1].w};
            uint16_t h[8], m[8], l[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                bad |= live && !isfinite(v[k]);
                split3(live ? v[k] : 0.0f, h[k], m[k], l[k]);
            }
            auto pack = [](const uint16_t *t) {
                return __builtin_bit_cast(bf16x8, make_uint4(t[0] | (uint32_t)t[1] << 16,
                                                             t[2] | (uint32_t)t[3] << 16,
                                                             t[4] | (uint32_t)t[5] << 16,
                                                             t[6] | (uint32_t)t[7] << 16));
            };
            mfma_block(acc, w, u, pack(h), pack(m), pack(l), kb0 + u < kb_end);
        }
    }
    partial[wave * 64 + lane] = acc;
    __syncthreads();
    if (wave == 0) {
        f32x4 v = acc;
#pragma unroll
        for (int w = 1; w < kTaskWaves; w++) {
            const f32x4 p = partial[w * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = __fadd_rn(v[r], p[r]);
        }
        EpiOperands e;
        load_epilogue_static<EPI_STORE>(e, a, s, row0, live);
        bad |= epilogue<EPI_STORE>(a, e, v, s, row0, live);
    }
    flag_nonfinite(a.status, bad);
}

template <int SRC, int EPI, bool Q8>
static int launch(const GemmArgs &a, hipStream_t stream) {
    if (a.n_rows <= 0 || a.n_rows % 16 || a.k_cols <= 0 || a.k_cols % 32 || a.streams <= 0 ||
        (SRC != SRC_SPLIT && a.k_cols != kWidth))
        return bad_arguments("pgpu_gemm");
    if constexpr (SRC != SRC_SPLIT) {
        const dim3 grid((a.n_rows / 16 + 3) / 4, (a.streams + 15) / 16);
        hipLaunchKernelGGL((k_gemm_wide<SRC, EPI, Q8>), grid, dim3(kTaskThreads), 0, stream, a);
    } else {
        const dim3 grid(a.n_rows / 16, (a.streams + 15) / 16);
        hipLaunchKernelGGL((k_gemm<EPI, Q8>), grid, dim3(kTaskThreads), 0, stream, a);
    }
    return launch_ok("pgpu_gemm");
}

template <int EPI>
static int dispatch(const GemmArgs &a, int q8, hipStream_t stream) {
    if (a.plain_rows)
        return q8 ? launch<SRC_ROWS, EPI, true>(a, stream)
                  : launch<SRC_ROWS, EPI, false>(a, stream);
    const int src = a.ln_x ? SRC_LN : (a.part_acc ? SRC_ATTN : SRC_SPLIT);
    if (src == SRC_LN)
        return q8 ? launch<SRC_LN, EPI, true>(a, stream) : launch<SRC_LN, EPI, false>(a, stream);
    if (src == SRC_ATTN)
        return q8 ? launch<SRC_ATTN, EPI, true>(a, stream)
                  : launch<SRC_ATTN, EPI, false>(a, stream);
    return q8 ? launch<SRC_SPLIT, EPI, true>(a, stream)
              : launch<SRC_SPLIT, EPI, false>(a, stream);
}

// Fills the operand-source fields from a pgpu_gemm_input.
static bool set_input(GemmArgs &a, const pgpu_gemm_input *in) {
    if (!in) return false;
    const int kinds = (in->split != nullptr) + (in->ln_rows != nullptr) +
                      (in->attn_acc != nullptr) + (in->rows != nullptr);
    if (kinds != 1) return false;
    a.xs = in->split;
    a.ln_x = in->rows ? in->rows : in->ln_rows;
    a.plain_rows = in->rows != nullptr;
    a.ln_w = in->ln_weight;
    a.ln_b = in->ln_bias;
    a.ln_eps = in->ln_epsilon;
    a.part_acc = in->attn_acc;
    a.part_ml = in->attn_ml;
    a.max_splits = in->attn_max_splits;
    if (in->ln_rows && (!a.ln_w || !a.ln_b)) return false;
    if (a.part_acc && (!a.part_ml || a.max_splits <= 0 || !in->attn_positions)) return false;
    if (a.part_acc) a.positions = in->attn_positions;
    return true;
}

static bool base_args(GemmArgs &a, const pgpu_matrix *w, const pgpu_gemm_input *in, int streams,
                      int *status) {
    a = GemmArgs{};
    a.w = w->values;
    a.wscale = w->scales;
    a.n_rows = (int)w->rows;
    a.k_cols = (int)w->columns;
    a.streams = streams;
    a.status = status;
    return set_input(a, in);
}

}  // namespace pgpu

using namespace pgpu;

extern "C" int pgpu_gemm_store(void *stream, const pgpu_matrix *w, const pgpu_gemm_input *in,
                               int streams, const float *bias, float *out, int ld_out,
                               int *status) {
    GemmArgs a;
    if (!base_args(a, w, in, streams, status)) return bad_arguments("pgpu_gemm_store");
    a.out = out;
    a.ld_out = ld_out;
    a.bias = bias;
    return dispatch<EPI_STORE>(a, w->q8, (hipStream_t)stream);
}

extern "C" int pgpu_gemm_store_rows(void *stream, const pgpu_matrix *w, const float *rows,
                                    int streams, float *out, int ld_out, int *status) {
    GemmArgs a;
    const pgpu_gemm_input in = {.rows = rows};
    if (!w || !w->q8 || !rows || !out || !status || streams <= 0 || !w->rows || w->rows % 16 ||
        !w->columns || w->columns % 32 || !base_args(a, w, &in, streams, status))
        return bad_arguments("pgpu_gemm_store_rows");
    a.out = out;
    a.ld_out = ld_out;
    const dim3 grid(a.n_rows / 16, (streams + 15) / 16);
    // A wave's blocks in equal chunks of at most 8 (a block past its range costs
    // what a block costs).
    const int per = (a.k_cols / 32 + kTaskWaves - 1) / kTaskWaves, chunks = (per + 7) / 8;
    const int ch = (per + chunks - 1) / chunks;
    const auto k = ch <= 1   ? k_gemm_rows<1>
                   : ch <= 2 ? k_gemm_rows<2>
                   : ch <= 4 ? k_gemm_rows<4>
                   : ch <= 6 ? k_gemm_rows<6>
                             : k_gemm_rows<8>;
    hipLaunchKernelGGL(k, grid, dim3(kTaskThreads), 0, (hipStream_t)stream, a);
    return launch_ok("pgpu_gemm_store_rows");
}

extern "C" int pgpu_gemm_residual(void *stream, const pgpu_matrix *w, const pgpu_gemm_input *in,
                                  int streams, const float *residual, float *out, int *status) {
    GemmArgs a;
    if (!base_args(a, w, in, streams, status)) return bad_arguments("pgpu_gemm_residual");
    a.out = out;
    a.ld_out = (int)w->rows;
    a.residual = residual;
    return dispatch<EPI_RESIDUAL>(a, w->q8, (hipStream_t)stream);
}

extern "C" int pgpu_gemm_gelu_split(void *stream, const pgpu_matrix *w,
                                    const pgpu_gemm_input *in, int streams, uint16_t *out_split,
                                    int *status) {
    GemmArgs a;
    if (!base_args(a, w, in, streams, status)) return bad_arguments("pgpu_gemm_gelu_split");
    a.out_split = out_split;
    a.out_kb = (int)w->rows / 32;
    return dispatch<EPI_GELU_SPLIT>(a, w->q8, (hipStream_t)stream);
}

extern "C" int pgpu_gemm_silu_split(void *stream, const pgpu_matrix *w,
                                    const pgpu_gemm_input *in, int streams, const float *bias,
                                    const float *bias2, uint16_t *out_split, int *status) {
    GemmArgs a;
    if (w->rows % 32 || !base_args(a, w, in, streams, status))
        return bad_arguments("pgpu_gemm_silu_split");
    a.bias = bias;
    a.bias2 = bias2;
    a.out_split = out_split;
    a.out_kb = (int)w->rows / 32;
    return dispatch<EPI_SILU_SPLIT>(a, w->q8, (hipStream_t)stream);
}

extern "C" int pgpu_gemm_gated(void *stream, const pgpu_matrix *w, const pgpu_gemm_input *in,
                               int streams, const float *bias, const float *gate, int ld_gate,
                               const float *residual, float *out, int *status) {
    GemmArgs a;
    if (!gate || !residual || (ld_gate != 0 && ld_gate < (int)w->rows) || ld_gate % 4 ||
        !base_args(a, w, in, streams, status))
        return bad_arguments("pgpu_gemm_gated");
    a.bias = bias;
    a.gate = gate;
    a.ld_gate = ld_gate;
    a.residual = residual;
    a.out = out;
    a.ld_out = (int)w->rows;
    return dispatch<EPI_GATED>(a, w->q8, (hipStream_t)stream);
}

extern "C" int pgpu_gemm_qkv(void *stream, const pgpu_matrix *w, const pgpu_gemm_input *in,
                             int streams, const pgpu_paged_kv *kv, int layer,
                             const int32_t *tables, int table_stride, const int32_t *positions,
                             const float *rope, float *q_out, int *status) {
    GemmArgs a;
    if (w->rows != 3 * kWidth || w->columns != kWidth || layer < 0 || layer >= kv->layers ||
        !base_args(a, w, in, streams, status) || a.part_acc)
        return bad_arguments("pgpu_gemm_qkv");
    a.q_out = q_out;
    a.kv = kv->base;
    a.layer_stride = kv->layer_stride;
    a.blocks = (unsigned)kv->blocks;
    a.layer = layer;
    a.tables = tables;
    a.table_stride = table_stride;
    a.positions = positions;
    a.rope = (const float2 *)rope;
    return dispatch<EPI_QKV>(a, w->q8, (hipStream_t)stream);
}
