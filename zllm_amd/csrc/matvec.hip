// Decode multiplies: out[t][col0 + j] (+)= sum_i X(t, i) * w[j][i] for Q8_0,
// Q3_K, Q4_K, Q5_K, Q6_K and BF16 weights, with the RMSNorm / activation prologues and the
// accumulate / SiLU-pair epilogues of the reference's matvec kernels
// (src/kernels/matvec_quant.wgsl.hbs:20-31, src/kernels/matvec_half.wgsl:14-19).
//
// General kernel. A workgroup is four wave64s. The step's inputs are staged
// once per workgroup in LDS (normalised / activated as they are staged), then
// every wave walks row groups in a grid-stride loop: a group is two weight
// rows (two outputs, or the gate and up rows of one output with SILU_PAIR).
// A row's packed weights are split into 16-byte tasks across the 64 lanes, so
// each load instruction of a wave reads consecutive 16-byte vectors; a lane
// decodes its task's weights once and multiplies them with every token's
// inputs; the lanes' partial sums reduce in a fixed butterfly. A token's sums
// are therefore the same bit for bit whether it runs alone or with others
// (the reference's split invariant, matvec_quant.wgsl.hbs:14-18).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "decode.h"
#include "matvec_common.h"

namespace zhip {

// The 16-bit formats' tasks are eight weights against two neighbouring input vectors. Lanes
// reading vector 2 task (then 2 task + 1) of a token would touch every other 16 bytes of LDS,
// two lanes to a bank; their inputs are therefore staged with the even vectors first and the
// odd ones behind them, so that each read covers consecutive vectors.
template <class D> constexpr bool kSplitInputs = std::is_same<D, DecBF16>::value || std::is_same<D, DecF16>::value;

// DEPTH: positions of the 16-bit formats' walk whose loads are in flight behind the one multiplied.
template <class D, int MT, int DEPTH>
__global__ __launch_bounds__(256) void matvec_kernel(MvArgs a) {
    extern __shared__ float4 xs4[];
    float *xs = reinterpret_cast<float *>(xs4);
    __shared__ float red[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t gwave = blockIdx.x * 4u + wave, nwaves = gridDim.x * 4u;
    const bool pair = (a.flags & FLAG_SILU_PAIR) != 0;
    const uint32_t k4 = a.k / 4u;
    const uint32_t tasks = a.k / D::E;
    // Outputs per group: two rows, or one gate/up pair.
    const uint32_t per_group = pair ? 1u : 2u;
    const uint32_t groups = (a.rows + per_group - 1u) / per_group;

    for (uint32_t t0 = 0; t0 < a.m; t0 += MT) {
        const uint32_t mt = min((uint32_t)MT, a.m - t0);
        __syncthreads();
        if constexpr (kSplitInputs<D>) {
            // The 16-bit formats. With rows of up to 4096 weights the pass's inputs are loaded
            // first (up to four vectors a thread and token, four tokens at a time), then the
            // wave's first weights, and only then are the inputs staged: the one trip to memory
            // serves both, where staging token after token and then starting on the weights
            // took one for every token and one more (loads complete in order within a wave).
            // A wave walks (group, 64-task slice) positions with the loads of the next DEPTH
            // positions in flight while it multiplies the current one (past its last position
            // the loads are clamped to a valid one and their data unused).
            constexpr int TG = MT < 4 ? MT : 4;
            // (a lone token gets here with longer rows only: matvec_half_row.hip takes the others)
            const bool early = MT > 1 && a.k <= 4096u;
            const uint32_t iters = (tasks + 63u) / 64u;
            auto place = [k4](uint32_t i) { return (i & 1u) * (k4 / 2u) + (i >> 1); };
            float4 xv[TG][4], gv[4];
            auto load_tokens = [&](uint32_t first) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t i = tid + 256u * j;
#pragma unroll
                    for (int t = 0; t < TG; t++) {
                        const float4 *xrow = reinterpret_cast<const float4 *>(a.x + (size_t)(t0 + (first + t < mt ? first + t : 0u)) * a.xr);
                        xv[t][j] = i < k4 ? xrow[i] : make_float4(0.f, 0.f, 0.f, 0.f);
                    }
                }
            };
            if (early) {
                load_tokens(0);
                if (a.flags & FLAG_NORM) {
                    const float4 *nw = reinterpret_cast<const float4 *>(a.norm_w);
#pragma unroll
                    for (int j = 0; j < 4; j++) gv[j] = tid + 256u * j < k4 ? nw[tid + 256u * j] : make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
            auto rows_of = [&](uint32_t g, uint32_t &j0, uint32_t &r1, bool &has1) {
                j0 = pair ? g : 2u * g;
                r1 = pair ? a.half + g : j0 + 1u;
                has1 = pair || r1 < a.rows;
            };
            auto load_at = [&](uint32_t g, uint32_t it, uint4 &q0, uint4 &q1) {
                uint32_t j0, r1;
                bool has1;
                rows_of(g < groups ? g : groups - 1u, j0, r1, has1);
                const uint32_t task = lane + 64u * it, tk = task < tasks ? task : 0u;
                q0 = *reinterpret_cast<const uint4 *>(a.w + (size_t)j0 * a.row_bytes + 16u * tk);
                q1 = *reinterpret_cast<const uint4 *>(a.w + (size_t)(has1 ? r1 : j0) * a.row_bytes + 16u * tk);
            };
            auto advance = [&](uint32_t &g, uint32_t &it) {
                if (++it == iters) {
                    it = 0;
                    g += nwaves;
                }
            };
            uint4 b0[DEPTH], b1[DEPTH];
            uint32_t lg = gwave, lit = 0;
#pragma unroll
            for (int s = 0; s < DEPTH; s++) {
                load_at(lg, lit, b0[s], b1[s]);
                advance(lg, lit);
            }
            if (early) {
                // The arithmetic of stage_token on the vectors already loaded, in the same
                // order, the tokens' sums of squares meeting in LDS together.
#pragma unroll
                for (int first = 0; first < MT; first += TG) {
                    if (first > 0) load_tokens(first);
                    float scale[TG];
#pragma unroll
                    for (int t = 0; t < TG; t++) scale[t] = 1.0f;
                    if (a.flags & FLAG_NORM) {
                        float ss[TG];
#pragma unroll
                        for (int t = 0; t < TG; t++) {
                            ss[t] = 0.f;
#pragma unroll
                            for (int j = 0; j < 4; j++)
                                if (tid + 256u * j < k4) ss[t] += xv[t][j].x * xv[t][j].x + xv[t][j].y * xv[t][j].y + xv[t][j].z * xv[t][j].z + xv[t][j].w * xv[t][j].w;
                            ss[t] = wave_sum(ss[t]);
                        }
                        __syncthreads();
                        if (lane == 0) {
#pragma unroll
                            for (int t = 0; t < TG; t++) red[4 * t + wave] = ss[t];
                        }
                        __syncthreads();
#pragma unroll
                        for (int t = 0; t < TG; t++) {
                            const float total = (red[4 * t] + red[4 * t + 1]) + (red[4 * t + 2] + red[4 * t + 3]);
                            scale[t] = 1.0f / sqrtf(total / (float)a.k + a.eps);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < TG; t++) {
                        float4 *dst = xs4 + (size_t)(first + t) * k4;
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const uint32_t i = tid + 256u * j;
                            if (i >= k4) continue;
                            float4 v = xv[t][j];
                            if (a.flags & FLAG_NORM) {
                                v.x = v.x * scale[t] * gv[j].x; v.y = v.y * scale[t] * gv[j].y;
                                v.z = v.z * scale[t] * gv[j].z; v.w = v.w * scale[t] * gv[j].w;
                            }
                            if (a.act_div > 0.f) {
                                v.x = silu_f(v.x / a.act_div); v.y = silu_f(v.y / a.act_div);
                                v.z = silu_f(v.z / a.act_div); v.w = silu_f(v.w / a.act_div);
                            }
                            if ((uint32_t)(first + t) >= mt) v = make_float4(0.f, 0.f, 0.f, 0.f);  // (a pass of fewer tokens than it has room for)
                            dst[place(i)] = v;
                        }
                    }
                }
            } else {
                for (uint32_t t = 0; t < (uint32_t)MT; t++) {
                    float4 *dst = xs4 + (size_t)t * k4;
                    if (t >= mt) {
                        for (uint32_t i = tid; i < k4; i += 256u) dst[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                        continue;
                    }
                    stage_token(a, t0 + t, dst, red, place);
                }
            }
            __syncthreads();

            float acc0[MT], acc1[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) acc0[t] = acc1[t] = 0.f;
            uint32_t g = gwave, it = 0;
            while (g < groups) {
#pragma unroll
                for (int s = 0; s < DEPTH; s++) {
                    if (g >= groups) break;
                    const uint4 c0 = b0[s], c1 = b1[s];
                    load_at(lg, lit, b0[s], b1[s]);
                    advance(lg, lit);
                    const uint32_t task = lane + 64u * it;
                    if (task < tasks) {
                        float w0[D::E], w1[D::E];
                        D::expand(c0, w0);
                        D::expand(c1, w1);
#pragma unroll
                        for (int t = 0; t < MT; t++) {
                            const float *xt = xs + (size_t)t * a.k;
                            float s0 = 0.f, s1 = 0.f;
#pragma unroll
                            for (int h = 0; h < 2; h++) {
                                const float4 v = *reinterpret_cast<const float4 *>(xt + 4u * ((uint32_t)h * (k4 / 2u) + task));
                                const int b = 4 * h;
                                s0 = fmaf(w0[b + 0], v.x, s0); s1 = fmaf(w1[b + 0], v.x, s1);
                                s0 = fmaf(w0[b + 1], v.y, s0); s1 = fmaf(w1[b + 1], v.y, s1);
                                s0 = fmaf(w0[b + 2], v.z, s0); s1 = fmaf(w1[b + 2], v.z, s1);
                                s0 = fmaf(w0[b + 3], v.w, s0); s1 = fmaf(w1[b + 3], v.w, s1);
                            }
                            acc0[t] += s0;
                            acc1[t] += s1;
                        }
                    }
                    if (it + 1u == iters) {
                        uint32_t j0, r1;
                        bool has1;
                        rows_of(g, j0, r1, has1);
#pragma unroll
                        for (int t = 0; t < MT; t++) {
                            acc0[t] = wave_sum(acc0[t]);
                            acc1[t] = wave_sum(acc1[t]);
                        }
                        if (lane == 0) {
                            for (uint32_t t = 0; t < mt; t++) {
                                const size_t o = (size_t)(t0 + t) * a.out_stride + a.col0 + j0;
                                if (pair) {
                                    float v = silu_f(acc0[t]) * acc1[t];
                                    if (a.flags & FLAG_ACCUMULATE) v += a.out[o];
                                    a.out[o] = v;
                                } else {
                                    float v = acc0[t];
                                    if (a.flags & FLAG_ACCUMULATE) v += a.out[o];
                                    a.out[o] = v;
                                    if (has1) {
                                        float u = acc1[t];
                                        if (a.flags & FLAG_ACCUMULATE) u += a.out[o + 1];
                                        a.out[o + 1] = u;
                                    }
                                }
                            }
                        }
#pragma unroll
                        for (int t = 0; t < MT; t++) acc0[t] = acc1[t] = 0.f;
                    }
                    advance(g, it);
                }
            }
            continue;
        }
        for (uint32_t t = 0; t < (uint32_t)MT; t++) {
            float4 *dst = xs4 + (size_t)t * k4;
            if (t >= mt) {
                for (uint32_t i = tid; i < k4; i += 256u) dst[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                continue;
            }
            stage_token(a, t0 + t, dst, red);
        }
        __syncthreads();
        for (uint32_t g = gwave; g < groups; g += nwaves) {
            // The group's two weight rows and whether each exists.
            const uint32_t j0 = pair ? g : 2u * g;
            const uint32_t r1 = pair ? a.half + g : j0 + 1u;
            const bool has1 = pair || r1 < a.rows;
            const uint8_t *row0 = a.w + (size_t)j0 * a.row_bytes;
            const uint8_t *row1 = a.w + (size_t)(has1 ? r1 : j0) * a.row_bytes;
            float acc0[MT], acc1[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) acc0[t] = acc1[t] = 0.f;

            for (uint32_t task = lane; task < tasks; task += 64u) {
                float w0[D::E], w1[D::E];
                D::decode(row0, a.k, task, w0);
                D::decode(row1, a.k, task, w1);
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const float *xt = xs + (size_t)t * a.k;
                    float s0 = 0.f, s1 = 0.f;
#pragma unroll
                    for (int h = 0; h < D::RUNS; h++) {
                        const float4 *xv = reinterpret_cast<const float4 *>(xt + D::xoff(task, h));
#pragma unroll
                        for (int e = 0; e < D::E / (4 * D::RUNS); e++) {
                            const float4 v = xv[e];
                            const int b = h * (D::E / D::RUNS) + 4 * e;
                            s0 = fmaf(w0[b + 0], v.x, s0); s1 = fmaf(w1[b + 0], v.x, s1);
                            s0 = fmaf(w0[b + 1], v.y, s0); s1 = fmaf(w1[b + 1], v.y, s1);
                            s0 = fmaf(w0[b + 2], v.z, s0); s1 = fmaf(w1[b + 2], v.z, s1);
                            s0 = fmaf(w0[b + 3], v.w, s0); s1 = fmaf(w1[b + 3], v.w, s1);
                        }
                    }
                    acc0[t] += s0;
                    acc1[t] += s1;
                }
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                acc0[t] = wave_sum(acc0[t]);
                acc1[t] = wave_sum(acc1[t]);
            }
            if (lane == 0) {
                for (uint32_t t = 0; t < mt; t++) {
                    const size_t o = (size_t)(t0 + t) * a.out_stride + a.col0 + j0;
                    if (pair) {
                        float v = silu_f(acc0[t]) * acc1[t];
                        if (a.flags & FLAG_ACCUMULATE) v += a.out[o];
                        a.out[o] = v;
                    } else {
                        float v = acc0[t];
                        if (a.flags & FLAG_ACCUMULATE) v += a.out[o];
                        a.out[o] = v;
                        if (has1) {
                            float u = acc1[t];
                            if (a.flags & FLAG_ACCUMULATE) u += a.out[o + 1];
                            a.out[o + 1] = u;
                        }
                    }
                }
            }
        }
    }
}

// The matrix-core variant of the quantized formats, any row length (matvec_mfma_rows.hip) ...
bool matvec_mfma_rows_accepts(const MvArgs &a);
zhip_result launch_matvec_mfma_rows(const Dispatch &d, const MvArgs &a, int type);
// ... and the kernels that are the faster ones on some shapes: Q4_K and Q5_K over rows of 2048 weights, or 6144 ..
// 32768 in parts of 2048 (matvec_mfma_resident.hip), Q8_0 over the same (matvec_q8_mfma_stream.hip), Q6_K, Q3_K and
// Q8_0 over long walks of tiles (matvec_q6k_mfma_stream.hip).
bool matvec_q4k_mfma_resident_accepts(const MvArgs &a);
zhip_result launch_matvec_q4k_mfma_resident(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
bool matvec_q5k_mfma_resident_accepts(const MvArgs &a);
zhip_result launch_matvec_q5k_mfma_resident(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
bool matvec_q8_mfma_stream_accepts(const MvArgs &a);
zhip_result launch_matvec_q8_mfma_stream(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
bool matvec_q6k_mfma_stream_accepts(const MvArgs &a);
zhip_result launch_matvec_q6k_mfma_stream(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
bool matvec_q3k_mfma_stream_accepts(const MvArgs &a);
zhip_result launch_matvec_q3k_mfma_stream(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
bool matvec_q8_0_mfma_flat_accepts(const MvArgs &a);
zhip_result launch_matvec_q8_0_mfma_flat(const Dispatch &d, const MvArgs &a, uint64_t w_bytes);
// Which of them takes a matrix under the matrix-core id: a property of the launch's matrix (type, row length, its rows, pair or not) and of
// the device's compute units, never of the step, since they add in
// different orders and a token's bits must not depend on the width of its step. us at one / four / eight
// tokens, weights from HBM, these kernels / matvec_mfma_rows.hip:
//  * Q4_K, Q5_K, Q8_0, rows of 2048 weights: Q4_K 4096 outputs 6.8 6.8 6.9 / 6.7 7.2 8.0, 2 x 8192 10.1 10.0 10.2 / 9.8
//    10.4 11.1, Q8_0 4096 6.9 7.0 7.1 / 7.1 7.5 8.1. Not rows of 4096: Q4_K 4096 outputs 10.3 10.3 10.8 / 6.9 7.7 10.0,
//    2 x 14336 21.7 21.2 21.8 / 19.7 19.5 21.4, Q5_K 27.5 27.7 28.3 / 22.4 22.0 24.5, Q8_0 4096 10.9 10.8 11.3 / 7.8 8.1 10.2. (Without RMSNorm
//    eight tokens over many rows pay for one to four: Q4_K 2 x 14336 20.1 20.0 19.9 / 19.5 18.3 20.5, Q8_0 14336 15.6 15.5 16.0 / 15.7 15.5 16.5.)
//  * the same in parts of 2048, no gate / up pair (and of Q8_0 fewer than 8192 outputs): at four tokens the two are within 5 % of each other on most, at eight
//    matvec_mfma_rows.hip is up to 40 % behind over few rows. Q4_K 2560 x 8192 9.8 9.8 9.9 / 10.4 11.0 13.1, 4096 x 8192 11.1 10.9 11.5 / 10.8 11.3 13.4, 4096 x 14336
//    15.0 14.8 15.4 / 13.8 14.2 16.4, 16384 x 8192 21.8 22.0 22.8 / 20.9 21.1 23.4, Q5_K 4096 x 6144 12.2 12.2 12.4 / 11.2 11.8 14.0, 16384 x 14336 41.9 41.9 43.0 / 38.5 38.7 41.2,
//    Q3_K 4096 x 6144 12.8 12.7 13.3 / 11.2 11.4 13.1, 16384 x 6144 22.9 22.6 24.1 / 24.4 24.7 26.8, Q8_0 2560 x 8192 10.8 10.9 11.2 / 11.4 12.1 13.3,
//    4096 x 14336 18.7 18.9 19.4 / 17.1 18.1 18.9; past the line Q8_0 8192 x 6144 17.2 17.6 18.0 / 14.6 15.3 17.7, 16384 x 8192 32.7 33.7 34.8 / 27.6 28.5 30.5.
//    Pairs: Q4_K 2 x 8192 x 8192 26.7 27.3 27.6 / 21.4 22.2 26.6, 2 x 14336 x 14336 61.0 62.2 62.9 / 52.6 55.2 55.8 (2 x 14336 x 6144 pays at eight, 32.1 32.6 32.9 / 30.2 31.9 36.8),
//    Q8_0 2 x 8192 x 8192 37.2 38.0 39.0 / 27.7 28.8 31.4.
//  * Q6_K, Q3_K and Q8_0 rows of 1024 weights: from twelve tiles of sixteen outputs a CU on (Q3_K: eight). Q6_K (rows of 1024
//    weights always: 4096 outputs 7.3 7.2 7.3 / 6.6 7.1 7.7) 64000 x 4096 (four and eight tokens) 46.4 49.7 / 51.2 52.9, 32000 x 4096 28.6 29.6 / 28.7 30.6, 4096 x 4096 14.7 15.5 /
//    8.6 10.3; Q3_K 64000 x 4096 38.9 40.9 / 42.9 44.1, 28672 x 4096 23.4 25.4 / 22.1 24.2, 4096 x 4096 12.7 13.3 / 7.4 9.4;
//    Q8_0 151936 x 1024 33.1 33.2 / 36.1 36.0, 50257 x 1024 16.9 16.8 / 16.7 16.8, 2 x 3072 x 1024 9.0 9.1 / 7.3 7.9, 4096 x 1024 (one, four, eight) 7.3 7.3 7.4 / 6.4 6.9
//    7.5, 1024 x 1024 6.7 6.8 6.9 / 5.9 6.5 7.2.
//  * Q3_K rows of 1024 weights, no pair: but where the tiles of a CU fill matvec_mfma_rows.hip's rounds of four. 4096 outputs 6.4 6.4 6.5 /
//    6.6 7.1 7.7, 9000 7.9 8.0 8.2 / 9.1 9.7 10.2, 16384 (four a CU) 8.3 8.3 8.6 / 7.3 7.2 7.5, 20480 9.4 9.4 9.7 / 9.7 9.6 9.9, 24576 9.4 9.3 9.6 / 9.9 9.6 10.0,
//    32000 (eight) 10.9 11.0 11.5 / 10.3 10.0 10.4.
//  * Q6_K in parts, no pair: from four tiles a CU on. 4096 x 6144 14.7 14.7 15.4 / 11.9 12.5 14.1, 8192 x 8192 19.6 19.4 20.5 / 18.5 18.8 20.5,
//    8192 x 14336 28.2 28.2 30.3 / 28.0 27.8 30.0, 16384 x 6144 26.0 25.9 27.7 / 26.8 26.9 28.8, 16384 x 14336 43.8 44.1 47.4 / 46.9 47.3 50.5,
//    28672 x 14336 72.9 73.7 76.5 / 78.9 79.5 83.1; pairs 2 x 14336 x 6144 41.3 41.8 44.4 / 41.0 41.9 44.2, 2 x 14336 x 8192 46.2 46.6 49.6 / 44.2
//    45.3 48.3, 2 x 14336 x 14336 75.4 77.5 82.4 / 76.3 78.0 82.7.
//  * gate / up pairs from seven tiles a CU on (Q6_K: rows of 3072 and 4096 weights), other rows of 3072 weights earlier still (twelve blocks for sixteen waves). Q3_K 2 x 14336 x 4096 with
//    RMSNorm 23.7 23.4 25.2 / 24.6 24.6 26.9, without 22.1 21.8 23.7 / 24.3 24.0 25.8, 2 x 12288 x 4096 23.5 23.4 25.2 / 20.5 19.8 22.0,
//    2 x 14336 x 2048 15.0 15.0 16.1 / 15.4 15.8 16.3, 2 x 14336 x 6144 36.9 37.3 39.8 / 39.3 40.8 44.6; Q6_K 2 x 14336 x 4096 28.0 26.8 28.6 / 27.5 27.0 28.5,
//    without RMSNorm 26.0 25.1 26.8 / 27.2 26.8 28.1, 2 x 12288 x 4096 26.8 26.7 28.3 / 22.6 22.6 24.3. Rows of 3072: Q3_K 12288 outputs 14.7 14.5 15.3 /
//    12.1 12.3 14.6, 16384 14.5 14.3 15.1 / 14.4 14.7 16.9, 32000 20.2 20.2 21.5 / 23.9 24.5 26.8, 2 x 4096 14.2 13.9 14.7 / 9.5 9.9 12.0, 2 x 6144 14.4
//    14.1 14.9 / 14.6 14.9 17.1; Q6_K 20480 20.7 20.2 21.5 / 18.1 17.9 20.3, 24576 20.6 20.5 21.5 / 21.0 20.3 22.8, 32000 24.0 23.7 25.1 / 25.7 25.4 27.9, 2 x 12288 23.9 23.6 24.9 / 21.0 20.4 22.7.
static bool older_mfma_pays(const Dispatch &d, const MvArgs &a, int type) {
    const bool pair = a.flags & FLAG_SILU_PAIR, parts = a.k > 4096u;
    const uint64_t tiles = ((uint64_t)a.rows * (pair ? 2u : 1u) + 15u) / 16u, cus = (uint64_t)d.dev->compute_units;
    const uint64_t each = (tiles + cus - 1u) / cus;
    switch (type) {
    case 4: case 5: return a.k == 2048u || (parts && !pair);
    case 8: return a.k == 1024u ? tiles >= 12u * cus : a.k == 2048u || (parts && !pair && a.rows < 8192u);
    case 6: return a.k == 1024u || (parts ? !pair && tiles >= 4u * cus : tiles >= (pair && a.k >= 3072u ? 7u : a.k == 3072u ? 6u : 12u) * cus);
    default:
        if (a.k == 1024u) return pair ? tiles >= 8u * cus : tiles >= 8u * cus || !(each == 4u || each == 7u || each == 8u);
        if (a.k == 3072u) return tiles >= (pair ? 3u : 4u) * cus;
        return pair ? tiles >= 7u * cus : parts || tiles >= 8u * cus;
    }
}
// matvec_bf16 on the matrix cores, the weights read once for all tokens (matvec_bf16_mfma_stream.hip).
bool matvec_bf16_mfma_stream_accepts(const MvArgs &a);
zhip_result launch_matvec_bf16_mfma_stream(const Dispatch &d, const MvArgs &a, uint64_t w_bytes, bool f16);
// Which matrices take it: rows of whole 512s in matrices of 16 MB of weights or more, gate / up pairs of 32 MB or more,
// and without the RMSNorm prologue, from 4 MB on, every matrix of rows of 6400 weights or more (no pairs), in
// contexts opened with ZHIP_OPTION_WIDE_DECODE, and then at every width from one token on: the
// kernel sums in another order than the general one, and a token's bits must not depend on the
// width of the step it runs in (src/sched/sched.zig:55-58; src/plan/qwen35.zig:380-381), so the
// route is a property of the matrix and of the context, never of the step. Its time hardly
// depends on the width, so such a context has steps of eight tokens at the price of its one-token
// steps, and pays for them at one token and, up to 40 MB or so, at four. With the RMSNorm prologue, this
// kernel / a default context's (matvec_half_row.hip, and matvec_kernel past its registers) at 1, 2, 4, 8 tokens, f16:
//   4096 x 2048 (16 MB)          8.4 8.4 8.5 8.6 / 5.1 5.6 6.6 8.9 us
//   8192 x 2048                  11.0 11.0 10.9 11.1 / 7.3 8.0 9.9 13.3
//   4096 x 4096                  13.0 13.2 13.2 13.5 / 8.4 9.2 11.7 17.2
//   151936 x 1024                52.9 53.6 54.2 54.3 / 53.6 56.8 61.5 85.7
//   2 x 8192 x 1024 (32 MB)      9.5 9.5 9.5 9.5 / 8.5 9.1 11.3 16.2
//   2 x 4096 x 2048 (32 MB)      12.2 12.1 12.2 12.2 / 7.9 8.3 9.9 13.9
//   2 x 8192 x 2048              17.8 17.9 17.9 18.0 / 13.6 14.6 17.2 38.1
//   2 x 14336 x 4096             46.8 47.9 47.9 50.5 / 40.9 51.3 61.1 107
// and below the line, where only the default kernels run:
//   4096 x 1024 (8 MB)           3.9 4.0 4.5 5.9
//   2048 x 2048 (8 MB)           4.2 4.9 4.9 6.0
// Long rows are past the registers of matvec_half_row.hip, and the general kernel takes them two tokens a pass over the weights, above
// 8192 weights one. Without the prologue, this kernel / the general one at 1, 2, 4 tokens, f16, weights from memory:
//   344 x 6400 (4 MB)            9.8 9.9 10.0 / 7.2 9.7 16.6
//   983 x 6400                   11.1 11.1 11.2 / 8.2 10.8 17.7
//   3276 x 6400 (40 MB)          18.0 17.9 17.8 / 12.9 16.0 25.0
//   5980 x 6400                  23.3 23.4 23.4 / 19.1 26.0 40.1
//   273 x 8064 (4 MB)            9.0 9.0 9.0 / 7.8 10.7 18.8
//   2600 x 8064 (40 MB)          15.7 15.7 15.5 / 13.7 17.1 27.3
//   2184 x 9600                  17.8 17.9 17.9 / 15.3 23.6 40.9
//   191 x 11520 (4 MB)           10.3 10.4 10.5 / 10.2 17.2 31.0
//   1820 x 11520 (40 MB)         16.8 17.0 16.8 / 15.7 24.7 44.1
//   1285 x 16320 (40 MB)         15.6 15.6 15.5 / 20.5 33.0 58.6
// Over 160 matrices of 6400 ... 16320 weights a row, 4 ... 80 MB, three tokens take 0.4 - 0.8 of the general kernel's time, eight 0.2 - 0.4. Two are
// level at 6400 in small matrices (0.8 - 1.1 below 7300, at the worst 1.17 at 40 MB; 0.4 - 1.0 from 7700 on) and below that line slower, 1024 x
// 6144 11.3 / 11.3, 3200 x 5248 14.3 / 13.4: it lies where a step of two breaks even. One token pays 1.1 - 1.4 times the time up to
// 7500 weights (fifteen lines of 512 columns, which the stretches do not divide evenly), 0.9 - 1.3 up to 13056, less than the general
// kernel's from there on: less than it pays in the table above. Matrices of under 4 MB were not measured.
// Shorter rows of no multiple of 512 stay with matvec_half_row.hip, which is the faster one at one and two tokens, at two by up to
// 35 % (5376 x 1792 pair 13.3 / 9.5, 8064 x 2688 22.0 / 17.1; at eight 13.3 / 17.7, 22.5 / 31.6).
constexpr uint64_t kBf16StreamBytes = kMatvecBf16StreamBytes, kBf16StreamLongBytes = 4ull << 20;
constexpr uint32_t kBf16StreamLong = 6400u;
static bool bf16_stream_pays(const Dispatch &d, const MvArgs &a) {
    const uint64_t bytes = (uint64_t)a.rows * a.row_bytes;  // (of a pair: of its gate rows)
    if (a.k % 512u == 0 && bytes >= kBf16StreamBytes) return d.dev->wide_decode;
    return d.dev->wide_decode && a.k >= kBf16StreamLong && bytes >= kBf16StreamLongBytes && !(a.flags & FLAG_NORM);
}
// The 16-bit formats with the inputs in registers, one to eight tokens (matvec_half_row.hip).
bool matvec_half_row_accepts(const MvArgs &a);
zhip_result launch_matvec_half_row(const Dispatch &d, const MvArgs &a, bool f16);
// The tuned multiply (matvec_quant.h, a source file a format): type 3, 4, 5, 6 (K-quants) or 8 (Q8_0).
zhip_result launch_matvec_quant(const Dispatch &d, const MvArgs &a, int type);

template <class D, int MT>
static zhip_result run(const Dispatch &d, const MvArgs &a, uint32_t lds_bytes) {
    static bool configured[2] = {false, false};  // dynamic LDS above 64 KiB needs opting in once, kernel by kernel
    // Long rows of a matrix of few rows: a wave has few positions, each a trip to memory; four
    // in flight instead of one (1024 x 3072 bf16, eight tokens in passes of four: 9.0 -> 7.4 us a pass).
    // Elsewhere the registers that takes cost more than it gains (151936 x 1024: 52 -> 62 us).
    const bool deep = kSplitInputs<D> && a.k >= 2048u && (uint64_t)a.rows * a.row_bytes <= (64ull << 20);
    auto kernel = deep ? matvec_kernel<D, MT, kSplitInputs<D> ? 4 : 1> : matvec_kernel<D, MT, 1>;
    if (lds_bytes > 65536u && !configured[deep]) {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 64) != hipSuccess) {
            (void)hipGetLastError();
            return fail(d, ZHIP_E_BAD_COMMAND, "decode multiply: k = %u with %d tokens does not fit workgroup memory", a.k, MT);
        }
        configured[deep] = true;
    }
    const uint32_t per_group = (a.flags & FLAG_SILU_PAIR) ? 1u : 2u;
    const uint32_t groups = (a.rows + per_group - 1u) / per_group;
    const uint32_t want = (groups + 3u) / 4u;
    // Few enough workgroups that staging the inputs stays a small part of each
    // one's traffic, enough of them to keep every CU's SIMDs busy.
    const uint32_t cap = (uint32_t)d.dev->compute_units * (lds_bytes > 32768u ? 2u : 4u);
    const uint32_t blocks = want < cap ? want : cap;
    hipLaunchKernelGGL(kernel, dim3(blocks ? blocks : 1), dim3(256), lds_bytes, d.stream, a);
    return check_launch(d, D::name());
}

template <class D>
static zhip_result launch_matvec(const Dispatch &d, bool quant) {
    if (d.params_size < sizeof(MatvecParams)) return fail(d, ZHIP_E_BAD_COMMAND, "%s: params block of %zu bytes", D::name(), d.params_size);
    const MatvecParams &p = *reinterpret_cast<const MatvecParams *>(d.params);
    MatvecVariant v;
    if (quant && d.variant != 0) {
        v.wg = (d.variant & 0xffu) * 32u;
        v.lanes = (d.variant >> 8) & 0xffu;
        v.rows = (d.variant >> 16) & 0xffu;
        v.act_div = d.variant >> 24;
        if (v.wg == 0 || v.lanes == 0 || v.rows == 0 || v.wg % v.lanes != 0)
            return fail(d, ZHIP_E_BAD_COMMAND, "%s: variant id 0x%08x is not a MatvecVariant", D::name(), d.variant);
    }
    // Rows one workgroup of the logical grid covers (kernels.matvec_rows = 8
    // for the half-precision kernel, groupRows() for the quantized one).
    const uint32_t group_rows = quant ? v.groupRows() : 8u;
    if (d.grid[0] == 0 || d.grid[1] == 0 || d.grid[2] == 0) return ZHIP_OK;
    const uint64_t covered = (uint64_t)d.grid[0] * group_rows;
    MvArgs a{};
    a.n = p.n; a.k = p.k; a.col0 = p.col0; a.out_stride = p.out_stride; a.eps = p.eps;
    a.flags = p.flags; a.half = p.half;
    a.rows = (uint32_t)(covered < p.n ? covered : p.n);
    // The quantized kernel runs the first row of workgroups over up to
    // kMaxDecodeRows tokens; the half-precision one has a grid row per token.
    a.m = quant ? (d.grid[1] < kMaxDecodeRows ? d.grid[1] : kMaxDecodeRows) : d.grid[1];
    a.xr = (quant && p.x_stride != 0) ? p.x_stride * 4u : p.k;
    a.act_div = quant ? (float)v.act_div : 0.f;
    a.row_bytes = D::row_bytes(p.k);
    if (p.k == 0 || p.k % D::BLOCK != 0) return fail(d, ZHIP_E_BAD_COMMAND, "%s: k = %u is not a multiple of %u", D::name(), p.k, D::BLOCK);
    if (p.flags & ~7u) return fail(d, ZHIP_E_BAD_COMMAND, "%s: unknown flags 0x%x", D::name(), p.flags);
    if (a.rows == 0) return ZHIP_OK;
    const bool norm = p.flags & FLAG_NORM, pair = p.flags & FLAG_SILU_PAIR;
    for (int b = 1; b <= (norm ? 4 : 3); b++)
        if (!d.bind[b].bound) return fail(d, ZHIP_E_BAD_COMMAND, "%s: binding %d is not bound", D::name(), b);
    const uint64_t x_need = ((uint64_t)(a.m - 1) * a.xr + p.k) * 4u;
    const uint64_t w_rows = pair ? (uint64_t)p.half + a.rows : a.rows;
    const uint64_t w_need = w_rows * a.row_bytes;
    const uint64_t o_need = ((uint64_t)(a.m - 1) * p.out_stride + p.col0 + a.rows) * 4u;
    if (x_need > d.bind[1].size) return fail(d, ZHIP_E_BAD_COMMAND, "%s: x needs %llu bytes, %llu bound", D::name(), (unsigned long long)x_need, (unsigned long long)d.bind[1].size);
    if (w_need > d.bind[2].size) return fail(d, ZHIP_E_BAD_COMMAND, "%s: weights need %llu bytes, %llu bound", D::name(), (unsigned long long)w_need, (unsigned long long)d.bind[2].size);
    if (o_need > d.bind[3].size) return fail(d, ZHIP_E_BAD_COMMAND, "%s: out needs %llu bytes, %llu bound", D::name(), (unsigned long long)o_need, (unsigned long long)d.bind[3].size);
    if (norm && (uint64_t)p.k * 4u > d.bind[4].size) return fail(d, ZHIP_E_BAD_COMMAND, "%s: norm weights need %u bytes", D::name(), p.k * 4u);
    if (((uintptr_t)d.bind[1].ptr | (uintptr_t)d.bind[2].ptr | (norm ? (uintptr_t)d.bind[4].ptr : 0)) & 15u)
        return fail(d, ZHIP_E_BAD_COMMAND, "%s: x, weights and norm weights must be 16-byte aligned", D::name());
    if (((uintptr_t)d.bind[3].ptr & 3u) || (a.xr & 3u)) return fail(d, ZHIP_E_BAD_COMMAND, "%s: misaligned out or x stride", D::name());
    a.x = reinterpret_cast<const float *>(d.bind[1].ptr);
    a.w = d.bind[2].ptr;
    a.out = reinterpret_cast<float *>(d.bind[3].ptr);
    a.norm_w = norm ? reinterpret_cast<const float *>(d.bind[4].ptr) : nullptr;

    // matvec_bf16 / matvec_f16 over a matrix of some size, in a context that asked for it, go to
    // the kernel that reads the weights once for all of a step's tokens.
    if ((std::is_same<D, DecBF16>::value || std::is_same<D, DecF16>::value) && bf16_stream_pays(d, a) && matvec_bf16_mfma_stream_accepts(a))
        return launch_matvec_bf16_mfma_stream(d, a, d.bind[2].size, std::is_same<D, DecF16>::value);
    // Everything else of a few tokens over rows that fit the registers; the general kernel, with its
    // inputs in LDS, adds in the same order and lost on every shape measured (figures there).
    if (kSplitInputs<D> && matvec_half_row_accepts(a)) return launch_matvec_half_row(d, a, std::is_same<D, DecF16>::value);

    // MatvecVariant (wg 512, lanes 64, rows 16) names the matrix-core variants: sixteen rows a tile.
    // A matrix of up to eight million weights runs the default kernels under that id too: its
    // launch is over before the matrix cores' sixteen-row tiles have their operands built. us at 1 / 4 / 8 tokens,
    // matrix cores / default: Q8_0 1024 x 3072 5.8 6.4 8.1 / 3.2 4.3 5.8, Q4_K 4096 x 1792 6.5 7.0 8.0 / 3.9 5.6 7.8,
    // Q3_K 2560 x 2560 6.5 7.2 9.0 / 4.3 7.0 9.1, Q6_K 6.8 7.5 9.5 / 4.4 7.1 9.8; above, Q4_K 4096 x 4096 6.9 7.4 7.7 /
    // 5.7 8.1 11.2. Not so rows of whole 2048s, in Q8_0, Q6_K and Q3_K of 1024 and in Q6_K and Q3_K of 3072: the matrix cores' sums are the ones nearer to the
    // exact (relative error, matrix cores / default: at 1024 weights Q8_0 1.15e-7 / 1.36e-7, Q3_K 1.13e-7 / 2.13e-7, Q6_K 1.05e-7 /
    // 2.22e-7, at 3072 Q3_K 0.90e-7 / 1.96e-7, Q6_K 1.06e-7 / 2.05e-7), and callers of the id have always had them there.
    // Q4_K and Q5_K rows of 1024 weights want sixteen million weights (four tiles a CU: a round of the kernel's four teams). Q4_K
    // 4096 outputs 6.3 6.8 7.6 / 3.2 4.1 5.4, 9000 8.1 8.7 9.5 / 3.8 6.1 8.0, 11718 8.0 8.8 9.6 / 3.9 6.3 9.2, 16384 6.9 6.9 7.6 / 4.4 7.4 11.0.
    const uint64_t weights = (uint64_t)a.rows * a.k * (pair ? 2u : 1u);
    constexpr bool Q36 = D::CHUNK == 3 || D::CHUNK == 6, Q45 = D::CHUNK == 4 || D::CHUNK == 5;
    const bool always = a.k % 2048u == 0 || (a.k == 1024u && !Q45) || (a.k == 3072u && Q36);
    const bool small = !always && weights <= (Q45 && a.k == 1024u ? 12u << 20 : 8u << 20);
    const bool matrix_cores = quant && v.lanes == 64u && v.rows == 16u && !small && (D::CHUNK == 4 || D::CHUNK == 8 || D::CHUNK == 6 || D::CHUNK == 5 || D::CHUNK == 3);
    if (matrix_cores) {
        const bool rows = matvec_mfma_rows_accepts(a), older = !rows || older_mfma_pays(d, a, D::CHUNK);
        if (D::CHUNK == 4 && older && matvec_q4k_mfma_resident_accepts(a)) return launch_matvec_q4k_mfma_resident(d, a, d.bind[2].size);
        if (D::CHUNK == 5 && older && matvec_q5k_mfma_resident_accepts(a)) return launch_matvec_q5k_mfma_resident(d, a, d.bind[2].size);
        if (D::CHUNK == 6 && older && matvec_q6k_mfma_stream_accepts(a)) return launch_matvec_q6k_mfma_stream(d, a, d.bind[2].size);
        if (D::CHUNK == 3 && older && matvec_q3k_mfma_stream_accepts(a)) return launch_matvec_q3k_mfma_stream(d, a, d.bind[2].size);
        if (D::CHUNK == 8 && older && matvec_q8_0_mfma_flat_accepts(a)) return launch_matvec_q8_0_mfma_flat(d, a, d.bind[2].size);
        if (D::CHUNK == 8 && older && matvec_q8_mfma_stream_accepts(a)) return launch_matvec_q8_mfma_stream(d, a, d.bind[2].size);
        if (rows) return launch_matvec_mfma_rows(d, a, D::CHUNK);
    }
    // The tuned kernel takes rows of whole 64-weight tasks.
    if (D::CHUNK != 0 && p.k % 64u == 0) return launch_matvec_quant(d, a, D::CHUNK);

    // Tokens per pass over the weights: as many as fit workgroup memory.
    const uint64_t row_lds = (uint64_t)p.k * 4u;
    const uint64_t max_lds = 160u * 1024u - 64u;
    uint32_t mt = a.m >= 5 ? 8u : a.m >= 3 ? 4u : a.m;
    while (mt > 1 && mt * row_lds > 65536u) mt >>= 1;
    if (mt * row_lds > max_lds) return fail(d, ZHIP_E_BAD_COMMAND, "%s: k = %u does not fit workgroup memory", D::name(), p.k);
    const uint32_t lds = (uint32_t)(mt * row_lds);
    switch (mt) {
    case 1: return run<D, 1>(d, a, lds);
    case 2: return run<D, 2>(d, a, lds);
    case 4: return run<D, 4>(d, a, lds);
    default: return run<D, 8>(d, a, lds);
    }
}

zhip_result launch_matvec_q8_0(const Dispatch &d) { return launch_matvec<DecQ8_0>(d, true); }
zhip_result launch_matvec_q4_k(const Dispatch &d) { return launch_matvec<DecQ4_K>(d, true); }
zhip_result launch_matvec_q3_k(const Dispatch &d) { return launch_matvec<DecQ3_K>(d, true); }
zhip_result launch_matvec_q5_k(const Dispatch &d) { return launch_matvec<DecQ5_K>(d, true); }
zhip_result launch_matvec_q6_k(const Dispatch &d) { return launch_matvec<DecQ6_K>(d, true); }
zhip_result launch_matvec_bf16(const Dispatch &d) { return launch_matvec<DecBF16>(d, false); }
zhip_result launch_matvec_f16(const Dispatch &d) { return launch_matvec<DecF16>(d, false); }

}  // namespace zhip
