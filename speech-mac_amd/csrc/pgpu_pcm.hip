// The latent-to-PCM decoder (src/phonon_mimi.c, src/phonon_pcm.c:145-170).
// Mimi's two layers are six launches each (LayerNorm, in-projection with RoPE
// and the ring, attention, out-projection, LayerNorm, the two MLP
// projections), the SEANet half seven: conv0, then per stage a transposed
// convolution and its residual pair, the output convolution inside the last
// pair.
//
// What bounds it. Every product is fp32-accurate: a bf16 weight times the
// three exact bf16 terms of an fp32 value, three matrix products. Splitting
// a value (and its ELU) costs about 25 vector instructions, so it is done
// once, where the value is produced (planes buffers), or once per work-group
// that needs all of a position's channels anyway (the residual pairs, whose
// hidden rows never leave LDS). A kernel that split its input for every tap
// and column tile was bound by those instructions: its eleven launches took
// 240 us per 32 frames and 155 us for one, these take 92 and 46 us. Mimi's
// layers, with 16-position projection tiles and an attention on the vector
// units before, went from 165 to 118 us per 32 frames and from 74 to 66 for one.
//
// Order of summation. k_plane_product sums a fixed four ranges of input
// channels (one wave each; within one, 32-channel block by block, its taps in
// order) and adds the four in order; the residual kernel runs one chain. No
// output depends on the tile shape or on how many positions a pass has, so a
// request gives the same bits however it is cut into calls.
#include "pgpu_gemm.hpp"
#include "pgpu_pcm.h"

namespace pgpu {
namespace {

constexpr int kSlots = 8;  // slots before a planes buffer's own positions

__device__ inline float elu1(float v) { return v <= 0.0f ? expf(v) - 1.0f : v; }

__device__ inline uint32_t pack16(uint16_t a, uint16_t b) { return a | (uint32_t)b << 16; }

// Four consecutive channels (c % 4 == 0) of position t as the planes' three
// terms.
__device__ inline void store_planes4(const pgpu_planes &out, int t, int c, const float *v) {
    uint16_t h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; i++) split3(v[i], h[i], m[i], l[i]);
    const uint2 term[3] = {{pack16(h[0], h[1]), pack16(h[2], h[3])},
                           {pack16(m[0], m[1]), pack16(m[2], m[3])},
                           {pack16(l[0], l[1]), pack16(l[2], l[3])}};
    const int octets = out.channels >> 3;
#pragma unroll
    for (int i = 0; i < 3; i++)
        ((uint2 *)out.data)[((size_t)(i * octets + (c >> 3)) * out.stride + kSlots + t) * 2 +
                            ((c >> 2) & 1)] = term[i];
}

// A wave normalises two rows with the decode step's LayerNorm arithmetic;
// lane j holds channels 8j .. 8j + 7, a slot of each term. Four waves write
// eight consecutive slots.
__global__ __launch_bounds__(256) void k_ln_planes(const float *__restrict__ rows,
                                                   const float *__restrict__ lw,
                                                   const float *__restrict__ lb, float eps,
                                                   int positions, pgpu_planes out, int *status) {
    const int j = threadIdx.x & 63, t0 = blockIdx.x * 8 + (threadIdx.x >> 6) * 2;
    Rows2 r;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        r.live[i] = t0 + i < positions;
        const float *src = rows + (size_t)(r.live[i] ? t0 + i : positions - 1) * kWidth + j * 8;
        const float4 a = *(const float4 *)src, b = *(const float4 *)(src + 4);
        r.v[i][0] = a.x; r.v[i][1] = a.y; r.v[i][2] = a.z; r.v[i][3] = a.w;
        r.v[i][4] = b.x; r.v[i][5] = b.y; r.v[i][6] = b.z; r.v[i][7] = b.w;
    }
    const bool bad = rows_ln_values(r, lw, lb, eps);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        if (!r.live[i]) continue;
        uint16_t h[8], m[8], l[8];
#pragma unroll
        for (int e = 0; e < 8; e++) split3(r.v[i][e], h[e], m[e], l[e]);
        uint4 *dst = (uint4 *)out.data + (size_t)j * out.stride + kSlots + t0 + i;
        const size_t term = (size_t)(kWidth / 8) * out.stride;
        dst[0] = uint4{pack16(h[0], h[1]), pack16(h[2], h[3]), pack16(h[4], h[5]),
                       pack16(h[6], h[7])};
        dst[term] = uint4{pack16(m[0], m[1]), pack16(m[2], m[3]), pack16(m[4], m[5]),
                          pack16(m[6], m[7])};
        dst[2 * term] = uint4{pack16(l[0], l[1]), pack16(l[2], l[3]), pack16(l[4], l[5]),
                              pack16(l[6], l[7])};
    }
    flag_nonfinite(status, bad);
}

// Windowed causal attention of one latent frame's 16 rows and one head per
// work-group (the contract of pgpu_mimi_attention). Both products run on the
// fp32 matrix cores, whose operand layouts need no shuffles between them:
// lane (g, n) = (lane / 16, lane % 16) of S^T = K Q^T holds keys 4g + r of
// query n, which is the operand of O^T = V^T P^T when its step r takes keys
// 4g + r. The window's up to 17 tiles of 16 keys go round the four waves;
// every K and V value is loaded straight into its operand register, all of
// them before the first product (one memory latency instead of one per
// 64-key chunk, each behind a barrier; the products on the vector units took
// most of 30 us per layer at 32 frames and 12 at one). Sums over the waves
// go through LDS in wave order, so a row's bits depend on its position only.
constexpr int kWaveTiles = 5;
static_assert(4 * kWaveTiles * 16 >= 256 + 15, "four waves hold a frame's key window");

template <bool PLANES>
__global__ __launch_bounds__(256) void k_window_attention(
    const float *__restrict__ q, int ld_q, long long first, const float *__restrict__ ring_k,
    const float *__restrict__ ring_v, int ring, int context, float *__restrict__ rows,
    pgpu_planes out, int *status) {
    __shared__ float red[2][4][16];
    __shared__ float4 part[4][4][64];
    const int f = blockIdx.x, head = blockIdx.y;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const long long p0 = first + 16LL * f;
    const long long kstart = p0 - (context - 1) > 0 ? p0 - (context - 1) : 0;
    const int nkeys = (int)(p0 + 16 - kstart);  // <= 256 + 15
    const int slot0 = (int)(kstart % ring);
    auto slot = [&](int key) {
        key = slot0 + (key < nkeys ? key : nkeys - 1);
        return (size_t)(key < ring ? key : key - ring) * kWidth + head * kHeadDim;
    };
    float4 qv[4], kv[kWaveTiles][4], vv[kWaveTiles][4];
    const float *qrow = q + (size_t)(16 * f + n) * ld_q + head * kHeadDim + 16 * g;
#pragma unroll
    for (int d = 0; d < 4; d++) qv[d] = *(const float4 *)(qrow + 4 * d);
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++) {
        const float *src = ring_k + slot((wave + 4 * i) * 16 + n) + 16 * g;
#pragma unroll
        for (int d = 0; d < 4; d++) kv[i][d] = *(const float4 *)(src + 4 * d);
    }
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            vv[i][r] = *(const float4 *)(ring_v + slot((wave + 4 * i) * 16 + 4 * g + r) + 4 * n);
    f32x4 s[kWaveTiles];
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < kWaveTiles; i++)
                s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(((const float *)&kv[i][d])[e],
                                                            ((const float *)&qv[d])[e], s[i], 0, 0,
                                                            0);
    // Masks and the softmax of query n.
    const long long p = p0 + n;
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const long long kp = kstart + (wave + 4 * i) * 16 + 4 * g + r;
            s[i][r] = kp <= p && kp > p - context ? s[i][r] * 0.125f : -INFINITY;
            mx = fmaxf(mx, s[i][r]);
        }
    mx = xor16_32_max(mx);
    if (lane < 16) red[0][wave][lane] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0][0][n], red[0][1][n]), fmaxf(red[0][2][n], red[0][3][n]));
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            s[i][r] = s[i][r] == -INFINITY ? 0.0f : expf(s[i][r] - mx);
            total += s[i][r];
        }
    total = xor16_32_sum(total);
    if (lane < 16) red[1][wave][lane] = total;
    f32x4 o[4];
#pragma unroll
    for (int d = 0; d < 4; d++) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kWaveTiles; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int d = 0; d < 4; d++)
                o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(((const float *)&vv[i][r])[d],
                                                            s[i][r], o[d], 0, 0, 0);
    // o[d][r]: dimension 16 g + 4 r + d of query n. Wave w finishes r = w.
#pragma unroll
    for (int r = 0; r < 4; r++)
        part[wave][r][lane] = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
    __syncthreads();
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float4 a = part[w][wave][lane];
        v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
    }
    total = ((red[1][0][n] + red[1][1][n]) + red[1][2][n]) + red[1][3][n];
    const float inv = 1.0f / total;
    bool bad = !(total > 0.0f);
#pragma unroll
    for (int d = 0; d < 4; d++) {
        v[d] *= inv;
        bad |= !isfinite(v[d]);
    }
    const int t = 16 * f + n, c = head * kHeadDim + 16 * g + 4 * wave;
    if constexpr (PLANES) {
        store_planes4(out, t, c, v);
    } else {
#pragma unroll
        for (int d = 0; d < 4; d++) rows[(size_t)t * kWidth + c + d] = v[d];
    }
    flag_nonfinite(status, bad);
}

// Orders one wave's LDS writes before its own later LDS reads: the hardware
// runs a wave's LDS instructions in order, the compiler must not reorder.
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A work-group computes 16 PT positions x 16 CT columns; its four waves take
// a quarter of the input channels each. A wave stages 32-channel blocks of
// its tile's rows (taps - 1 more than positions) in its own part of LDS,
// requests the next ones and their weights, and then runs every tap from there:
// tap j reads the same slots j rows further on, a 256-byte run per 16 lanes
// either way.
constexpr int taps_of(int epi) {
    return epi == PGPU_PLANE_ROWS ? 2 : epi == PGPU_PLANE_ELU ? 7 : 1;
}

// 32-channel blocks a wave stages at once. A projection's one tap gives a
// block too little work to hide the next one's latency (the MLP-out product,
// 16 blocks a wave, took 11 us for one frame block by block); its small tiles
// leave the registers and LDS for four. in.channels is a multiple of 512 then.
constexpr int stage_blocks(int epi, int pt) { return taps_of(epi) == 1 ? 4 / pt : 1; }

// Four results o (columns col .. col + 3 of position t) on their way out.
// True if one is not finite.
template <int EPI>
__device__ inline bool plane_epilogue(const pgpu_plane_product &a, int t, int col, float *o) {
    bool bad = false;
    if constexpr (EPI == PGPU_PLANE_ROWS || EPI == PGPU_PLANE_ELU) {
        const float4 b = *(const float4 *)(a.bias + col % a.cout);
        o[0] = __fadd_rn(o[0], b.x);
        o[1] = __fadd_rn(o[1], b.y);
        o[2] = __fadd_rn(o[2], b.z);
        o[3] = __fadd_rn(o[3], b.w);
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !isfinite(o[r]);
        if constexpr (EPI == PGPU_PLANE_ROWS) {
            *(float4 *)(a.rows + (size_t)t * a.ncols + col) =
                make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = elu1(o[r]);
            store_planes4(a.planes, t, col, o);
        }
    } else if constexpr (EPI == PGPU_PLANE_GELU) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            o[r] = gelu_erf(o[r]);
            bad |= !isfinite(o[r]);
        }
        store_planes4(a.planes, t, col, o);
    } else if constexpr (EPI == PGPU_PLANE_GATED) {
        float4 *at = (float4 *)(a.rows + (size_t)t * kWidth + col);
        const float4 s = *at, k = *(const float4 *)(a.gate + col);
        o[0] = __fadd_rn(s.x, __fmul_rn(k.x, o[0]));
        o[1] = __fadd_rn(s.y, __fmul_rn(k.y, o[1]));
        o[2] = __fadd_rn(s.z, __fmul_rn(k.z, o[2]));
        o[3] = __fadd_rn(s.w, __fmul_rn(k.w, o[3]));
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !isfinite(o[r]);
        *at = make_float4(o[0], o[1], o[2], o[3]);
        if (a.planes.data) store_planes4(a.planes, t, col, o);
    } else {
        const int part = col >> 9, c = col & 511;
        const long long pos = a.first + t;
        if (part < 2) {
            const float4 cs = *(const float4 *)(a.rope + (size_t)pos * 64 + (c & 63));
            const float v[4] = {o[0], o[1], o[2], o[3]};
            o[0] = __fsub_rn(__fmul_rn(v[0], cs.x), __fmul_rn(v[1], cs.y));
            o[1] = __fadd_rn(__fmul_rn(v[0], cs.y), __fmul_rn(v[1], cs.x));
            o[2] = __fsub_rn(__fmul_rn(v[2], cs.z), __fmul_rn(v[3], cs.w));
            o[3] = __fadd_rn(__fmul_rn(v[2], cs.w), __fmul_rn(v[3], cs.z));
        }
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !isfinite(o[r]);
        float *dst = part == 0 ? a.rows + (size_t)t * kWidth
                               : (part == 1 ? a.ring_k : a.ring_v) +
                                     (size_t)(pos % a.ring) * kWidth;
        *(float4 *)(dst + c) = make_float4(o[0], o[1], o[2], o[3]);
    }
    return bad;
}

template <int EPI, int PT, int CT>
__global__ __launch_bounds__(256) void k_plane_product(pgpu_plane_product a, pgpu_planes in,
                                                       int positions, int past, int *status) {
    constexpr int TAPS = taps_of(EPI), KS = stage_blocks(EPI, PT);
    constexpr int kRows = 16 * PT + TAPS - 1;
    constexpr int kPieces = 12 * KS * kRows;  // (block, term, octet of the block, row)
    constexpr int kLoads = (kPieces + 63) / 64;
    constexpr int kStage = kLoads * 64;
    constexpr int kParts = 4 * PT * CT * 64;
    static_assert(kLoads <= 32, "one bit of `zero` per load");
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
        const int to = piece / kRows, term = to % 12 >> 2;
        int r = t0 + piece % kRows - (TAPS - 1);
        r = r < positions ? r : positions - 1;
        at[i] = (term * octets + 4 * (cb0 + to / 12) + (to & 3)) * in.stride + kSlots + r;
        zero |= (uint32_t)(r < 0 && !past) << i;
    }
    const uint4 *src = (const uint4 *)in.data;
    const int step = 4 * KS * in.stride;
    uint4 next[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) next[i] = src[at[i]];
    f32x4 acc[PT][CT];
#pragma unroll
    for (int p = 0; p < PT; p++)
#pragma unroll
        for (int q = 0; q < CT; q++) acc[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 *wsrc = (const bf16x8 *)a.fragments + (size_t)ct0 * kbn * 64 + lane;
    bf16x8 wnext[KS][TAPS][CT];
    auto request_weights = [&](int cb) {
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
                for (int q = 0; q < CT; q++)
                    wnext[k][tap][q] = wsrc[(size_t)(q * kbn + tap * cbn + cb + k) * 64];
    };
    request_weights(cb0);
    for (int cb = cb0; cb < cb1; cb += KS) {
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < kLoads; i++)
            stage[i * 64 + lane] = (zero >> i) & 1 ? uint4{0, 0, 0, 0} : next[i];
        bf16x8 wa[KS][TAPS][CT];
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
                for (int q = 0; q < CT; q++) wa[k][tap][q] = wnext[k][tap][q];
        if (cb + KS < cb1) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) {
                at[i] += step;
                next[i] = src[at[i]];
            }
            request_weights(cb + KS);
        }
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int tap = 0; tap < TAPS; tap++)
#pragma unroll
                for (int term = 0; term < 3; term++) {
                    bf16x8 xs[PT];
#pragma unroll
                    for (int p = 0; p < PT; p++)
                        xs[p] = __builtin_bit_cast(
                            bf16x8, stage[((k * 3 + term) * 4 + (lane >> 4)) * kRows + p * 16 +
                                          (lane & 15) + tap]);
#pragma unroll
                    for (int p = 0; p < PT; p++)
#pragma unroll
                        for (int q = 0; q < CT; q++)
                            acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                wa[k][tap][q], xs[p], acc[p][q], 0, 0, 0);
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
        float o[4] = {s[0], s[1], s[2], s[3]};
        bad |= plane_epilogue<EPI>(a, t, col, o);
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
                    store_planes4(out, t, c, o);
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

// The last 8 positions of each convolution's input, and the status word.
__global__ __launch_bounds__(256) void k_keep(pgpu_kept keep, const int *__restrict__ status,
                                              int *__restrict__ seen) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) *seen = *status;
    if (i >= PGPU_KEPT_SLOTS) return;
    uint4 *dst = (uint4 *)keep.kept + i;
#pragma unroll
    for (int p = 0; p < PGPU_KEPT_PLANES; p++) {
        const pgpu_planes &in = keep.in[p];
        const int count = 3 * in.channels;  // slots: 8 of each (term, octet)
        if (i < count) {
            *dst = ((const uint4 *)in.data)[(size_t)(i >> 3) * in.stride + keep.positions[p] +
                                            (i & 7)];
            return;
        }
        i -= count;
    }
}

bool planes_ok(const pgpu_planes *p, int positions) {
    return p && p->data && p->channels > 0 && p->channels % 32 == 0 &&
           p->stride >= kSlots + positions &&
           (size_t)3 * (p->channels / 8) * p->stride < (size_t)0x7fffffff;
}

bool pass_ok(pgpu_pass p) { return (p.phase == 0 || p.phase == 1) && (p.past == 0 || p.past == 1); }

template <int EPI, int PT, int CT>
void launch_product(hipStream_t st, const pgpu_plane_product &a, const pgpu_planes &in,
                    int positions, pgpu_pass pass, int *status) {
    const dim3 grid((positions + 16 * PT - 1) / (16 * PT), a.ncols / (16 * CT));
    hipLaunchKernelGGL((k_plane_product<EPI, PT, CT>), grid, dim3(256), 0, st, a, in, positions,
                       pass.past, status);
}

// Short passes are bound by latency, long ones by what the work-groups read
// from L2: per reduction index a tile reads 2 bytes a column and 6 a position,
// so tiles are wide in columns, and a larger one is taken as soon as it
// leaves enough work-groups (us, 4 x 4 / 2 x 4 tiles: 512 positions, 1536
// columns, K = 1024 14.0 / 10.8 at 192 groups of the larger; 1024 positions,
// 2048 columns, K = 512 16.4 / 18.9 at 512). conv0's seven taps of weights
// would not fit the registers of a 64-column tile; 4 x 2 took 22.8 us at 1024
// positions, 2 x 2 takes 16.9.
template <int EPI>
void launch_tile(hipStream_t st, const pgpu_plane_product &a, const pgpu_planes &in,
                 int positions, pgpu_pass pass, int *status) {
    auto groups = [&](int pt, int ct) {
        return (long)((positions + 16 * pt - 1) / (16 * pt)) * (a.ncols / (16 * ct));
    };
    if constexpr (EPI == PGPU_PLANE_ELU) {
        if (groups(2, 2) >= 96)
            return launch_product<EPI, 2, 2>(st, a, in, positions, pass, status);
    } else {
        if (groups(4, 4) >= 384)
            return launch_product<EPI, 4, 4>(st, a, in, positions, pass, status);
        if (groups(2, 4) >= 160)
            return launch_product<EPI, 2, 4>(st, a, in, positions, pass, status);
        if (groups(1, 4) >= 96)
            return launch_product<EPI, 1, 4>(st, a, in, positions, pass, status);
    }
    launch_product<EPI, 1, 1>(st, a, in, positions, pass, status);
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

extern "C" int pgpu_pcm_keep(void *stream, const pgpu_kept *keep, const int *status, int *seen) {
    constexpr int channels[PGPU_KEPT_PLANES] = {512, 512, 256, 128};
    bool ok = keep && keep->kept && status && seen;
    for (int p = 0; ok && p < PGPU_KEPT_PLANES; p++)
        ok = keep->positions[p] >= 8 && planes_ok(&keep->in[p], keep->positions[p]) &&
             keep->in[p].channels == channels[p];
    if (!ok) return bad_arguments("pgpu_pcm_keep");
    hipLaunchKernelGGL(k_keep, dim3((PGPU_KEPT_SLOTS + 255) / 256), dim3(256), 0,
                       (hipStream_t)stream, *keep, status, seen);
    return launch_ok("pgpu_pcm_keep");
}

extern "C" int pgpu_pcm_wait(void *event) {
    if (hipEventSynchronize((hipEvent_t)event) == hipSuccess) return 1;
    pgpu_record_error("pgpu_pcm_wait: hipEventSynchronize failed");
    return 0;
}

extern "C" int pgpu_pcm_layer_norm(void *stream, const float *rows, const float *weight,
                                   const float *bias, float epsilon, int positions,
                                   const pgpu_planes *out, int *status) {
    if (!rows || !weight || !bias || !(epsilon > 0.0f) || positions <= 0 ||
        !planes_ok(out, positions) || out->channels != kWidth || !status)
        return bad_arguments("pgpu_pcm_layer_norm");
    hipLaunchKernelGGL(k_ln_planes, dim3((positions + 7) / 8), dim3(256), 0, (hipStream_t)stream,
                       rows, weight, bias, epsilon, positions, *out, status);
    return launch_ok("pgpu_pcm_layer_norm");
}

static bool attention_ok(const float *q, int rows, long long first, const float *ring_k,
                         const float *ring_v, int ring, int context, const int *status) {
    return q && rows > 0 && rows % 16 == 0 && rows <= 65535 && first >= 0 && ring_k && ring_v &&
           context > 0 && context <= 256 && ring >= rows + context - 1 && status;
}

extern "C" int pgpu_pcm_attention(void *stream, const float *q, int rows, long long first,
                                  const float *ring_k, const float *ring_v, int ring, int context,
                                  const pgpu_planes *out, int *status) {
    if (!attention_ok(q, rows, first, ring_k, ring_v, ring, context, status) ||
        !planes_ok(out, rows) || out->channels != kWidth)
        return bad_arguments("pgpu_pcm_attention");
    hipLaunchKernelGGL(k_window_attention<true>, dim3(rows / 16, kHeads), dim3(256), 0,
                       (hipStream_t)stream, q, kWidth, first, ring_k, ring_v, ring, context,
                       nullptr, *out, status);
    return launch_ok("pgpu_pcm_attention");
}

extern "C" int pgpu_mimi_attention(void *stream, const float *qkv, int rows, long long first,
                                   const float *ring_k, const float *ring_v, int ring,
                                   int context, float *out, int *status) {
    if (!attention_ok(qkv, rows, first, ring_k, ring_v, ring, context, status) || !out)
        return bad_arguments("pgpu_mimi_attention");
    hipLaunchKernelGGL(k_window_attention<false>, dim3(rows / 16, kHeads), dim3(256), 0,
                       (hipStream_t)stream, qkv, 3 * kWidth, first, ring_k, ring_v, ring, context,
                       out, pgpu_planes{}, status);
    return launch_ok("pgpu_mimi_attention");
}

static bool product_ok(const pgpu_plane_product *a, const pgpu_planes *in, int positions) {
    if (!a || !a->fragments || positions < 8 || !planes_ok(in, positions) || in->channels % 128 ||
        a->ncols <= 0 || a->ncols % 64 ||
        (long)(positions + 15) / 16 * (a->ncols / 16) > 0x7fffffL)
        return false;
    const bool planes = planes_ok(&a->planes, positions) && a->planes.channels == a->ncols;
    switch (a->epilogue) {
    case PGPU_PLANE_ROWS:
        return a->rows && a->bias && a->cout > 0 && a->cout % 64 == 0;
    case PGPU_PLANE_ELU:
        return planes && a->bias && a->cout > 0 && a->cout % 64 == 0;
    case PGPU_PLANE_GELU:
        return planes && in->channels % 512 == 0;
    case PGPU_PLANE_GATED:
        return a->rows && a->gate && a->ncols == kWidth && (!a->planes.data || planes) &&
               in->channels % 512 == 0;
    case PGPU_PLANE_QKV:
        return a->rows && in->channels % 512 == 0 && a->ncols == 3 * kWidth && a->rope && a->first >= 0 &&
               a->first + positions <= a->rope_positions && a->ring_k && a->ring_v &&
               a->ring >= positions;
    }
    return false;
}

extern "C" int pgpu_pcm_product(void *stream, const pgpu_plane_product *a, const pgpu_planes *in,
                                int positions, pgpu_pass pass, int *status) {
    if (!product_ok(a, in, positions) || !pass_ok(pass) || !status)
        return bad_arguments("pgpu_pcm_product");
    hipStream_t st = (hipStream_t)stream;
    switch (a->epilogue) {
    case PGPU_PLANE_ROWS:
        launch_tile<PGPU_PLANE_ROWS>(st, *a, *in, positions, pass, status);
        break;
    case PGPU_PLANE_ELU:
        launch_tile<PGPU_PLANE_ELU>(st, *a, *in, positions, pass, status);
        break;
    case PGPU_PLANE_GELU:
        launch_tile<PGPU_PLANE_GELU>(st, *a, *in, positions, pass, status);
        break;
    case PGPU_PLANE_GATED:
        launch_tile<PGPU_PLANE_GATED>(st, *a, *in, positions, pass, status);
        break;
    default:
        launch_tile<PGPU_PLANE_QKV>(st, *a, *in, positions, pass, status);
    }
    return launch_ok("pgpu_pcm_product");
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
        // (64-position groups: 21.1 us at 29,760 positions, these 18.4.)
        launch_residual<128, 2>(st, *w, x, positions, pass, history, out, pcm, status);
    } else {
        launch_residual<64, 4>(st, *w, x, positions, pass, history, out, pcm, status);
    }
    return launch_ok("pgpu_pcm_residual");
}
