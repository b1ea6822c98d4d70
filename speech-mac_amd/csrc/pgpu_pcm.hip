// The SEANet half of the latent-to-PCM decoder (src/phonon_pcm.c:145-170),
// seven launches a pass: conv0, then per stage a transposed convolution and
// its residual pair, the output convolution inside the last pair.
//
// What bounds it. Every product is fp32-accurate: a bf16 weight times the
// three exact bf16 terms of an fp32 value, three matrix products. Splitting
// a value (and its ELU) costs about 25 vector instructions, so it is done
// once, where the value is produced (planes buffers), or once per work-group
// that needs all of a position's channels anyway (the residual pairs, whose
// hidden rows never leave LDS). A kernel that split its input for every tap
// and column tile was bound by those instructions: its eleven launches took
// 240 us per 32 frames and 155 us for one, these take 92 and 46 us.
//
// Order of summation. k_conv_planes sums a fixed four ranges of input
// channels (one wave each; within one, 32-channel block by block, its taps in
// order) and adds the four in order; the residual kernel runs one chain. No
// output depends on the tile shape or on how many positions a pass has, so a
// request gives the same bits however it is cut into calls.
#include "pgpu_common.hpp"
#include "pgpu_pcm.h"

namespace pgpu {
namespace {

constexpr int kSlots = 16;  // slots before a planes buffer's own positions

__device__ inline float elu1(float v) { return v <= 0.0f ? expf(v) - 1.0f : v; }

__device__ inline uint32_t pack16(uint16_t a, uint16_t b) { return a | (uint32_t)b << 16; }

// Slot of position r >= -8 of the pass.
__device__ inline int slot_of(int r, int phase) {
    return r < 0 ? 8 * phase + 8 + r : kSlots + r;
}

// Four consecutive channels (c % 4 == 0) of position t as the planes' three
// terms; the last 8 positions also where the next pass finds its past.
__device__ inline void store_planes4(const pgpu_planes &out, int t, int positions, int phase,
                                     int c, const float *v) {
    uint16_t h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; i++) split3(v[i], h[i], m[i], l[i]);
    const uint2 term[3] = {{pack16(h[0], h[1]), pack16(h[2], h[3])},
                           {pack16(m[0], m[1]), pack16(m[2], m[3])},
                           {pack16(l[0], l[1]), pack16(l[2], l[3])}};
    const int octets = out.channels >> 3;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        uint2 *p = (uint2 *)out.data +
                   ((size_t)(i * octets + (c >> 3)) * out.stride) * 2 + ((c >> 2) & 1);
        p[(size_t)(kSlots + t) * 2] = term[i];
        if (t >= positions - 8)
            p[(size_t)slot_of(t - positions, 1 - phase) * 2] = term[i];
    }
}

__global__ __launch_bounds__(256) void k_rows_to_planes(const float *__restrict__ rows,
                                                        int positions, pgpu_planes out,
                                                        int phase) {
    // 16 positions x 16 groups of four channels per work-group.
    const int t = blockIdx.x * 16 + (threadIdx.x & 15);
    const int c = (blockIdx.y * 16 + (threadIdx.x >> 4)) * 4;
    if (t >= positions) return;
    const float4 v = *(const float4 *)(rows + (size_t)t * kWidth + c);
    const float a[4] = {v.x, v.y, v.z, v.w};
    store_planes4(out, t, positions, phase, c, a);
}

// Orders one wave's LDS writes before its own later LDS reads: the hardware
// runs a wave's LDS instructions in order, the compiler must not reorder.
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A work-group computes 16 PT positions x 16 CT columns; its four waves take
// a quarter of the input channels each. A wave stages one 32-channel block of
// its tile's rows (taps - 1 more than positions) in its own part of LDS,
// requests the next block and its weights, and then runs every tap from there:
// tap j reads the same slots j rows further on, a 256-byte run per 16 lanes
// either way.
template <int TAPS, int PT, int CT>
__global__ __launch_bounds__(256) void k_conv_planes(pgpu_plane_conv conv, pgpu_planes in,
                                                     int positions, int phase, int past,
                                                     float *__restrict__ rows, pgpu_planes out,
                                                     int *status) {
    constexpr int kRows = 16 * PT + TAPS - 1;
    constexpr int kPieces = 12 * kRows;  // (term, octet of the block, row)
    constexpr int kLoads = (kPieces + 63) / 64;
    constexpr int kStage = kLoads * 64;
    constexpr int kParts = 4 * PT * CT * 64;
    __shared__ uint4 lds[4 * kStage > kParts ? 4 * kStage : kParts];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t0 = blockIdx.x * 16 * PT, ct0 = blockIdx.y * CT;
    const int octets = in.channels >> 3, cbn = in.channels >> 5, kbn = TAPS * cbn;
    const int cb0 = wave * cbn / 4, cb1 = (wave + 1) * cbn / 4;
    uint4 *stage = lds + wave * kStage;
    int at[kLoads];
    uint32_t zero = 0;  // bit i: load i of this lane lies before the request
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        int piece = i * 64 + lane;
        piece = piece < kPieces ? piece : kPieces - 1;
        const int to = piece / kRows;
        int r = t0 + piece % kRows - (TAPS - 1);
        r = r < positions ? r : positions - 1;
        at[i] = ((to >> 2) * octets + 4 * cb0 + (to & 3)) * in.stride + slot_of(r, phase);
        zero |= (uint32_t)(r < 0 && !past) << i;
    }
    const uint4 *src = (const uint4 *)in.data;
    const int step = 4 * in.stride;
    uint4 next[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) next[i] = src[at[i]];
    f32x4 acc[PT][CT];
#pragma unroll
    for (int p = 0; p < PT; p++)
#pragma unroll
        for (int q = 0; q < CT; q++) acc[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 *wsrc = (const bf16x8 *)conv.fragments + (size_t)ct0 * kbn * 64 + lane;
    bf16x8 wnext[TAPS][CT];
#pragma unroll
    for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
        for (int q = 0; q < CT; q++)
            wnext[tap][q] = wsrc[(size_t)(q * kbn + tap * cbn + cb0) * 64];
    for (int cb = cb0; cb < cb1; cb++) {
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < kLoads; i++)
            stage[i * 64 + lane] = (zero >> i) & 1 ? uint4{0, 0, 0, 0} : next[i];
        bf16x8 wa[TAPS][CT];
#pragma unroll
        for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
            for (int q = 0; q < CT; q++) wa[tap][q] = wnext[tap][q];
        if (cb + 1 < cb1) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) {
                at[i] += step;
                next[i] = src[at[i]];
            }
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
                for (int q = 0; q < CT; q++)
                    wnext[tap][q] = wsrc[(size_t)(q * kbn + tap * cbn + cb + 1) * 64];
        }
        wave_lds_order();
#pragma unroll
        for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
            for (int term = 0; term < 3; term++) {
                bf16x8 xs[PT];
#pragma unroll
                for (int p = 0; p < PT; p++)
                    xs[p] = __builtin_bit_cast(
                        bf16x8, stage[(term * 4 + (lane >> 4)) * kRows + p * 16 + (lane & 15) +
                                      tap]);
#pragma unroll
                for (int p = 0; p < PT; p++)
#pragma unroll
                    for (int q = 0; q < CT; q++)
                        acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            wa[tap][q], xs[p], acc[p][q], 0, 0, 0);
            }
    }
    __syncthreads();
    f32x4 *part = (f32x4 *)lds;
#pragma unroll
    for (int p = 0; p < PT; p++)
#pragma unroll
        for (int q = 0; q < CT; q++) part[((wave * PT + p) * CT + q) * 64 + lane] = acc[p][q];
    __syncthreads();
    bool bad = false;
    for (int f = wave; f < PT * CT; f += 4) {
        const int t = t0 + f / CT * 16 + (lane & 15);
        const int col = (ct0 + f % CT) * 16 + 4 * (lane >> 4);
        if (t >= positions) continue;
        f32x4 s = part[f * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; w++) {
            const f32x4 o = part[(w * PT * CT + f) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) s[r] = __fadd_rn(s[r], o[r]);
        }
        const float4 b = *(const float4 *)(conv.bias + col % conv.cout);
        float o[4] = {__fadd_rn(s[0], b.x), __fadd_rn(s[1], b.y), __fadd_rn(s[2], b.z),
                      __fadd_rn(s[3], b.w)};
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !isfinite(o[r]);
        if constexpr (TAPS == 2) {
            *(float4 *)(rows + (size_t)t * conv.ncols + col) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = elu1(o[r]);
            store_planes4(out, t, positions, phase, col, o);
        }
    }
    flag_nonfinite(status, bad);
}

// One work-group: 16 PT positions of a residual pair, all channels. The rows
// (two more than positions, for conv3's taps) are read once, their ELU split
// into LDS; conv3's result, its ELU split, stays in LDS as conv1's operand.
// Every weight a wave needs is requested before the step that precedes its
// use (a short pass is a chain of memory latencies otherwise). C = 64 ends
// with the decoder's output convolution: its ELU'd rows stay in LDS too, and
// a work-group writes 16 PT - 2 samples (its first two rows are only taps of
// the others).
constexpr int kResWaves = 8;

template <int C, int PT>
__global__ __launch_bounds__(64 * kResWaves) void k_residual(
    pgpu_residual_weights w, const float *__restrict__ x, int positions, int phase, int past,
    float *__restrict__ history, pgpu_planes out, float *__restrict__ pcm, int *status) {
    constexpr bool kLast = C == 64;
    constexpr int kT = 16 * PT, kRows = kT + 2, kHalf = C / 2;
    constexpr int kX = 3 * (C / 8) * kRows, kH = 3 * (kHalf / 8) * kT;
    __shared__ uint4 lds[kX + kH];
    __shared__ float4 last4[kLast ? 48 : 1];
    uint4 *xs = lds, *hs = lds + kX;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t0 = kLast ? blockIdx.x * (kT - 2) - 2 : blockIdx.x * kT;  // first residual row
    const float *before = history + (size_t)phase * 4 * C;  // rows -4 .. -1
    auto row = [&](int r) {
        r = r < positions ? r : positions - 1;
        return r < 0 ? before + (4 + r) * C : x + (size_t)r * C;
    };
    // conv3: a wave takes kQ3 column tiles and kP3 position tiles; conv1
    // kQ1 and kP1.
    constexpr int kWc3 = kHalf / 16 < kResWaves ? kHalf / 16 : kResWaves;
    constexpr int kQ3 = kHalf / 16 / kWc3, kP3 = PT * kWc3 / kResWaves;
    constexpr int kWc1 = C >= 256 ? kResWaves : 4;
    constexpr int kQ1 = C / 16 / kWc1, kP1 = PT * kWc1 / kResWaves;
    static_assert(kP3 >= 1 && kP1 >= 1, "every wave has a tile");
    constexpr int cbn = C / 32, kbn3 = 3 * cbn, kbn1 = kHalf / 32;
    const int q3 = wave % kWc3 * kQ3, p3 = wave / kWc3 * kP3;
    const int q1 = wave % kWc1 * kQ1, p1 = wave / kWc1 * kP1;
    bf16x8 w3[kbn3][kQ3];
    {
        const bf16x8 *src = (const bf16x8 *)w.conv3 + (size_t)q3 * kbn3 * 64 + lane;
#pragma unroll
        for (int kb = 0; kb < kbn3; kb++)
#pragma unroll
            for (int q = 0; q < kQ3; q++) w3[kb][q] = src[(q * kbn3 + kb) * 64];
    }
    // Rows t0 - 2 .. t0 + kT - 1: a wave takes 16 rows x 4 octets at a time.
    constexpr int kBlocks = (kRows + 15) / 16 * (C / 32);
    constexpr int kPer = (kBlocks + kResWaves - 1) / kResWaves;
    float4 in[kPer][2];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int b = i * kResWaves + wave;
        const int j = b / (C / 32) * 16 + (lane & 15), octet = b % (C / 32) * 4 + (lane >> 4);
        const float4 *src = (const float4 *)(row(t0 - 2 + j) + octet * 8);
        in[i][0] = src[0];
        in[i][1] = src[1];
    }
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < 4 * C; i += 64 * kResWaves)
            history[(size_t)(1 - phase) * 4 * C + i] = x[(size_t)(positions - 4) * C + i];
    if (kLast && threadIdx.x < 192) {
        const int i = threadIdx.x;  // tap * 64 + channel: record, lane 16 g, element
        ((float *)last4)[i] =
            bitsf((uint32_t)w.last[(i >> 5) * 512 + ((i >> 3) & 3) * 128 + (i & 7)] << 16);
    }
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int b = i * kResWaves + wave;
        const int j = b / (C / 32) * 16 + (lane & 15), octet = b % (C / 32) * 4 + (lane >> 4);
        if (b < kBlocks && j < kRows) {
            const bool live = t0 - 2 + j >= 0 || past;
            const float v[8] = {in[i][0].x, in[i][0].y, in[i][0].z, in[i][0].w,
                                in[i][1].x, in[i][1].y, in[i][1].z, in[i][1].w};
            uint16_t h[8], m[8], l[8];
#pragma unroll
            for (int e = 0; e < 8; e++) split3(live ? elu1(v[e]) : 0.0f, h[e], m[e], l[e]);
            uint4 *dst = xs + octet * kRows + j;
            dst[0] = uint4{pack16(h[0], h[1]), pack16(h[2], h[3]), pack16(h[4], h[5]),
                           pack16(h[6], h[7])};
            dst[(C / 8) * kRows] = uint4{pack16(m[0], m[1]), pack16(m[2], m[3]),
                                         pack16(m[4], m[5]), pack16(m[6], m[7])};
            dst[2 * (C / 8) * kRows] = uint4{pack16(l[0], l[1]), pack16(l[2], l[3]),
                                             pack16(l[4], l[5]), pack16(l[6], l[7])};
        }
    }
    bf16x8 w1[kbn1][kQ1];
    {
        const bf16x8 *src = (const bf16x8 *)w.conv1 + (size_t)q1 * kbn1 * 64 + lane;
#pragma unroll
        for (int kb = 0; kb < kbn1; kb++)
#pragma unroll
            for (int q = 0; q < kQ1; q++) w1[kb][q] = src[(q * kbn1 + kb) * 64];
    }
    __syncthreads();
    bool bad = false;
    {
        f32x4 acc[kP3][kQ3];
#pragma unroll
        for (int p = 0; p < kP3; p++)
#pragma unroll
            for (int q = 0; q < kQ3; q++) acc[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int cb = 0; cb < cbn; cb++)
#pragma unroll
            for (int tap = 0; tap < 3; tap++)
#pragma unroll
                for (int term = 0; term < 3; term++)
#pragma unroll
                    for (int p = 0; p < kP3; p++) {
                        const bf16x8 v = __builtin_bit_cast(
                            bf16x8, xs[(term * (C / 8) + cb * 4 + (lane >> 4)) * kRows +
                                       (p3 + p) * 16 + (lane & 15) + tap]);
#pragma unroll
                        for (int q = 0; q < kQ3; q++)
                            acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                w3[tap * cbn + cb][q], v, acc[p][q], 0, 0, 0);
                    }
#pragma unroll
        for (int p = 0; p < kP3; p++)
#pragma unroll
            for (int q = 0; q < kQ3; q++) {
                const int c = (q3 + q) * 16 + 4 * (lane >> 4), j = (p3 + p) * 16 + (lane & 15);
                const float4 b = *(const float4 *)(w.bias3 + c);
                const float o[4] = {__fadd_rn(acc[p][q][0], b.x), __fadd_rn(acc[p][q][1], b.y),
                                    __fadd_rn(acc[p][q][2], b.z), __fadd_rn(acc[p][q][3], b.w)};
                uint16_t h[4], m[4], l[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    bad |= !isfinite(o[r]);
                    split3(elu1(o[r]), h[r], m[r], l[r]);
                }
                uint2 *dst = (uint2 *)(hs + (c >> 3) * kT + j) + ((c >> 2) & 1);
                dst[0] = uint2{pack16(h[0], h[1]), pack16(h[2], h[3])};
                dst[2 * (kHalf / 8) * kT] = uint2{pack16(m[0], m[1]), pack16(m[2], m[3])};
                dst[4 * (kHalf / 8) * kT] = uint2{pack16(l[0], l[1]), pack16(l[2], l[3])};
            }
    }
    float4 skip[kP1][kQ1];
#pragma unroll
    for (int p = 0; p < kP1; p++)
#pragma unroll
        for (int q = 0; q < kQ1; q++)
            skip[p][q] = *(const float4 *)(row(t0 + (p1 + p) * 16 + (lane & 15)) +
                                           (q1 + q) * 16 + 4 * (lane >> 4));
    __syncthreads();
    float *es = (float *)xs;  // C = 64: ELU(v) [kT][kE], over the rows no longer needed
    constexpr int kE = 68;    // 16 rows' float4 reads fall on 16 different bank groups
    static_assert(!kLast || kT * kE <= 4 * kX, "the output convolution's rows fit");
    {
        f32x4 acc[kP1][kQ1];
#pragma unroll
        for (int p = 0; p < kP1; p++)
#pragma unroll
            for (int q = 0; q < kQ1; q++) acc[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < kbn1; kb++)
#pragma unroll
            for (int term = 0; term < 3; term++)
#pragma unroll
                for (int p = 0; p < kP1; p++) {
                    const bf16x8 v = __builtin_bit_cast(
                        bf16x8, hs[(term * (kHalf / 8) + kb * 4 + (lane >> 4)) * kT +
                                   (p1 + p) * 16 + (lane & 15)]);
#pragma unroll
                    for (int q = 0; q < kQ1; q++)
                        acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[kb][q], v,
                                                                            acc[p][q], 0, 0, 0);
                }
#pragma unroll
        for (int p = 0; p < kP1; p++)
#pragma unroll
            for (int q = 0; q < kQ1; q++) {
                const int c = (q1 + q) * 16 + 4 * (lane >> 4);
                const int j = (p1 + p) * 16 + (lane & 15), t = t0 + j;
                const bool live = t < positions && (t >= 0 || past);
                const float4 b = *(const float4 *)(w.bias1 + c);
                const float4 s = skip[p][q];
                float o[4] = {__fadd_rn(s.x, __fadd_rn(acc[p][q][0], b.x)),
                              __fadd_rn(s.y, __fadd_rn(acc[p][q][1], b.y)),
                              __fadd_rn(s.z, __fadd_rn(acc[p][q][2], b.z)),
                              __fadd_rn(s.w, __fadd_rn(acc[p][q][3], b.w))};
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    bad |= live && !isfinite(o[r]);
                    o[r] = live ? elu1(o[r]) : 0.0f;
                }
                if constexpr (kLast)
                    *(float4 *)(es + j * kE + c) = make_float4(o[0], o[1], o[2], o[3]);
                else if (live)
                    store_planes4(out, t, positions, phase, c, o);
            }
    }
    if constexpr (kLast) {
        __syncthreads();
        // Sample t0 + 2 + j from rows j .. j + 2: eight lanes, 8 channels each.
        static_assert(kT * 8 == 64 * kResWaves, "eight lanes per row");
        const int j = threadIdx.x >> 3, part = threadIdx.x & 7, t = t0 + 2 + j;
        float sum = 0.0f;
        if (j < kT - 2) {
#pragma unroll
            for (int tap = 0; tap < 3; tap++)
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const float4 e = *(const float4 *)(es + (j + tap) * kE + part * 8 + c * 4);
                    const float4 k = last4[tap * 16 + part * 2 + c];
                    sum = fmaf(k.x, e.x, sum);
                    sum = fmaf(k.y, e.y, sum);
                    sum = fmaf(k.z, e.z, sum);
                    sum = fmaf(k.w, e.w, sum);
                }
        }
        sum += __shfl_xor(sum, 1);
        sum += __shfl_xor(sum, 2);
        sum += __shfl_xor(sum, 4);
        if (j < kT - 2 && t < positions && part == 0) {
            const float v = sum + w.bias_last[0];
            bad |= !isfinite(v);
            pcm[t] = v;
        }
    }
    flag_nonfinite(status, bad);
}

bool planes_ok(const pgpu_planes *p, int positions) {
    return p && p->data && p->channels > 0 && p->channels % 32 == 0 &&
           p->stride >= kSlots + positions &&
           (size_t)3 * (p->channels / 8) * p->stride < (size_t)0x7fffffff;
}

bool pass_ok(pgpu_pass p) { return (p.phase == 0 || p.phase == 1) && (p.past == 0 || p.past == 1); }

template <int TAPS, int PT, int CT>
void launch_conv(hipStream_t st, const pgpu_plane_conv &c, const pgpu_planes &in, int positions,
                 pgpu_pass pass, float *rows, const pgpu_planes &out, int *status) {
    const dim3 grid((positions + 16 * PT - 1) / (16 * PT), c.ncols / (16 * CT));
    hipLaunchKernelGGL((k_conv_planes<TAPS, PT, CT>), grid, dim3(256), 0, st, c, in, positions,
                       pass.phase, pass.past, rows, out, status);
}

// The largest tile that still leaves a work-group for (nearly) every CU:
// larger tiles read each weight and row fewer times, smaller ones spread a
// short pass over the chip.
template <int TAPS>
void launch_conv_tile(hipStream_t st, const pgpu_plane_conv &c, const pgpu_planes &in,
                      int positions, pgpu_pass pass, float *rows, const pgpu_planes &out,
                      int *status) {
    auto groups = [&](int pt, int ct) {
        return (long)((positions + 16 * pt - 1) / (16 * pt)) * (c.ncols / (16 * ct));
    };
    constexpr long kFill = 224;
    if (TAPS == 2 && groups(4, 4) >= kFill)
        launch_conv<2, 4, 4>(st, c, in, positions, pass, rows, out, status);
    else if (groups(4, 2) >= kFill)
        launch_conv<TAPS, 4, 2>(st, c, in, positions, pass, rows, out, status);
    else if (groups(2, 2) >= kFill)
        launch_conv<TAPS, 2, 2>(st, c, in, positions, pass, rows, out, status);
    else
        launch_conv<TAPS, 1, 1>(st, c, in, positions, pass, rows, out, status);
}

template <int C, int PT>
void launch_residual(hipStream_t st, const pgpu_residual_weights &w, const float *x, int positions,
                     pgpu_pass pass, float *history, const pgpu_planes &out, float *pcm,
                     int *status) {
    const int step = C == 64 ? 16 * PT - 2 : 16 * PT;
    hipLaunchKernelGGL((k_residual<C, PT>), dim3((positions + step - 1) / step),
                       dim3(64 * kResWaves), 0, st, w, x, positions, pass.phase, pass.past, history, out, pcm, status);
}

}  // namespace
}  // namespace pgpu

using namespace pgpu;

extern "C" int pgpu_pcm_rows_to_planes(void *stream, const float *rows, int positions,
                                       const pgpu_planes *out, pgpu_pass pass) {
    if (!rows || positions < 8 || !planes_ok(out, positions) || out->channels != kWidth ||
        !pass_ok(pass))
        return bad_arguments("pgpu_pcm_rows_to_planes");
    hipLaunchKernelGGL(k_rows_to_planes, dim3((positions + 15) / 16, kWidth / 64), dim3(256), 0,
                       (hipStream_t)stream, rows, positions, *out, pass.phase);
    return launch_ok("pgpu_pcm_rows_to_planes");
}

extern "C" int pgpu_pcm_conv(void *stream, const pgpu_plane_conv *c, const pgpu_planes *in,
                             int positions, pgpu_pass pass, float *rows, const pgpu_planes *planes,
                             int *status) {
    if (!c || !c->fragments || !c->bias || positions < 8 || !planes_ok(in, positions) ||
        in->channels % 128 || c->ncols <= 0 || c->ncols % 64 || c->cout <= 0 || c->cout % 64 ||
        !pass_ok(pass) || !status || (c->taps != 2 && c->taps != 7) || (c->taps == 2 && !rows) ||
        (c->taps == 7 && (!planes_ok(planes, positions) || planes->channels != c->ncols)) ||
        (long)(positions + 15) / 16 * (c->ncols / 16) > 0x7fffffL)
        return bad_arguments("pgpu_pcm_conv");
    hipStream_t st = (hipStream_t)stream;
    if (c->taps == 2)
        launch_conv_tile<2>(st, *c, *in, positions, pass, rows, pgpu_planes{}, status);
    else
        launch_conv_tile<7>(st, *c, *in, positions, pass, nullptr, *planes, status);
    return launch_ok("pgpu_pcm_conv");
}

extern "C" int pgpu_pcm_residual(void *stream, const pgpu_residual_weights *w, int channels,
                                 const float *x, int positions, pgpu_pass pass, float *history,
                                 const pgpu_planes *planes, float *pcm, int *status) {
    const bool last = channels == 64;
    if (!w || !w->conv3 || !w->conv1 || !w->bias3 || !w->bias1 || !x || positions < 8 ||
        !pass_ok(pass) || !history || !status ||
        (channels != 256 && channels != 128 && channels != 64) ||
        (last ? !w->last || !w->bias_last || !pcm
              : !planes_ok(planes, positions) || planes->channels != channels))
        return bad_arguments("pgpu_pcm_residual");
    hipStream_t st = (hipStream_t)stream;
    const pgpu_planes out = last ? pgpu_planes{} : *planes;
    if (channels == 256) {
        if (positions <= 16 * 256)
            launch_residual<256, 1>(st, *w, x, positions, pass, history, out, pcm, status);
        else
            launch_residual<256, 2>(st, *w, x, positions, pass, history, out, pcm, status);
    } else if (channels == 128) {
        if (positions <= 32 * 256)
            launch_residual<128, 2>(st, *w, x, positions, pass, history, out, pcm, status);
        else
            launch_residual<128, 4>(st, *w, x, positions, pass, history, out, pcm, status);
    } else {
        launch_residual<64, 4>(st, *w, x, positions, pass, history, out, pcm, status);
    }
    return launch_ok("pgpu_pcm_residual");
}
