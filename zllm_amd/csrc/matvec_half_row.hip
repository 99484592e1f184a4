// matvec_bf16 and matvec_f16 with the inputs in registers: steps of one to eight tokens over
// rows of up to 5120 weights. A workgroup takes as many of the tokens as a lane's registers hold
// the inputs of, or fewer (see launch), others the rest.
//
// Such a launch reads a few MB and lasts a few microseconds, most of them trips to memory one
// behind the other. Here there is one: the tokens' inputs and the norm weights are asked for
// first, then the wave's first rows (loads complete in order within a wave), the inputs are
// normalised and handed round through LDS while the weights arrive, and from then on a lane holds
// the inputs of its tasks (eight weights of a row, 64 tasks apart) and the loop nothing but
// loads of the next pass and the multiply of the current one. A pass's loads go through a
// buffer that begins at its first row and ends with the matrix: rows past the end and lanes
// without a task read zeros. The rows' sums over the wave never leave the registers
// (wave_sum), a pass's outputs are stored together, and what they hold, for an accumulating
// step, is asked for with the pass's weights.
//
// The arithmetic of matvec.hip's kernel, which takes every other shape, in its order: the
// staging, a task's eight multiply-adds, the lane's tasks in turn, the wave's sum. A token's
// bits are the same in both and at every width.
//
// Measured from a graph over different weights (bf16; before: matvec.hip's kernel):
//   2048 x 1024, RMSNorm, at 1 / 2 / 4 / 8 tokens   4.0 / 4.4 / 5.9 / 9.1 -> 2.7 / 3.1 / 3.7 / 4.1 us
//   1024 x 2048, accumulating, at 1 / 2 / 4 / 8     4.4 / 5.4 / 7.5 / 11.5 -> 3.2 / 3.6 / 3.9 / 4.6
//   2 x 3072 x 1024, RMSNorm, at 1 / 2 / 4 / 8      6.0 / 6.4 / 11.4 / 10.4 -> 4.4 / 4.8 / 6.0 / 8.5
//   1024 x 3072, accumulating, at 1 / 2             4.9 / 6.1 -> 3.6 / 4.0
//   2560 x 4096 / 4096 x 4096, one token            8.8 / 9.6 -> 6.3 / 8.1
//   2 x 8192 x 2048 / 2 x 9728 x 2560, one token    15.4 / 23.4 -> 13.0 / 18.5
//   2 x 5120 x 5120 / 2 x 13824 x 5120, one token   22.6 / 53.5 -> 19.9 / 50.5 (f16, three registers of whose
//                                                   pair do not fit: 22.9 / 53.3 -> 20.9 / 52.9)
//   151936 x 1024 (311 MB), one token               52.8 -> 52.2 (6.0 TB/s)
// Short launches are bound by the launch itself (about 2.3 us with nothing in it) and one trip to
// memory, long ones by HBM.
#include <hip/hip_runtime.h>

#include "common.h"
#include "decode.h"
#include "matvec_common.h"

namespace zhip {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ROWS: weight rows a wave multiplies in a pass (with PAIR half of them gate rows, half up rows). KEEP: the
// outputs of 64 / OUTS passes wait in the lanes for one store; see launch_iters.
template <class D, int MT, int ITERS, bool PAIR, int ROWS, bool KEEP>
__global__ __launch_bounds__(256, 2) void matvec_half_row_kernel(MV_FIRST) {
    MvArgs a = MV_TAKE_FIRST(MT, PAIR);
    extern __shared__ float4 xs4[];
    __shared__ float red[4 * MT];
    constexpr int OUTS = PAIR ? ROWS / 2 : ROWS, XV = (ITERS + 1) / 2;
    // A step of more tokens than the registers hold: workgroups of their own for every MT of them.
    a.x += (size_t)(MT * blockIdx.y) * a.xr;
    if (MT > 1) a.m -= MT * blockIdx.y;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t k4 = a.k / 4u, tasks = a.k / 8u;
    const uint32_t passes = (a.rows + OUTS - 1u) / OUTS;
    const uint32_t first = blockIdx.x * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)wave), nwaves = gridDim.x * 4u;

    float4 xv[MT][XV], gv[XV];
#pragma unroll
    for (int j = 0; j < XV; j++) {
        const uint32_t i = tid + 256u * j;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const float4 *xrow = reinterpret_cast<const float4 *>(a.x + (size_t)t * a.xr);
            xv[t][j] = i < k4 && (uint32_t)t < a.m ? xrow[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    if (a.flags & FLAG_NORM) {
        const float4 *nw = reinterpret_cast<const float4 *>(a.norm_w);
#pragma unroll
        for (int j = 0; j < XV; j++) gv[j] = tid + 256u * j < k4 ? nw[tid + 256u * j] : make_float4(0.f, 0.f, 0.f, 0.f);
    }

    // Within a pass's buffer: the lane's task of the last 64 may lie past the row.
    const uint32_t at = 16u * lane, last_at = lane + 64u * (ITERS - 1) < tasks ? at : kNowhere;
    const uint64_t span = (uint64_t)a.rows * a.row_bytes;
    const bool accumulate = (a.flags & FLAG_ACCUMULATE) != 0;
    struct Pass {
        u32x4 q[ROWS][ITERS];
        float before[MT];
    };
    auto out_at = [&](int t, uint32_t j) __attribute__((always_inline)) { return a.out + (size_t)(MT * blockIdx.y + t) * a.out_stride + j; };
    auto fetch = [&](uint32_t u, Pass &p) __attribute__((always_inline)) {
        const bool live = u < passes;
        const uint64_t off = live ? (uint64_t)u * OUTS * a.row_bytes : 0u;
        const int left = live ? (int)(span - off) : 0;
        const __amdgpu_buffer_rsrc_t gate = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.w + off), 0, left, 0x00020000);
        const __amdgpu_buffer_rsrc_t up = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.w + (PAIR ? (uint64_t)a.half * a.row_bytes : 0u) + off), 0, left, 0x00020000);
#pragma unroll
        for (int r = 0; r < ROWS; r++)
#pragma unroll
            for (int it = 0; it < ITERS; it++)
                p.q[r][it] = __builtin_amdgcn_raw_buffer_load_b128(PAIR && r >= OUTS ? up : gate, (it == ITERS - 1 ? last_at : at) + (uint32_t)(PAIR && r >= OUTS ? r - OUTS : r) * a.row_bytes + 1024u * it, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // (the loads stay ahead of the multiply that follows them in the source)
        const uint32_t j = u * OUTS + lane;
#pragma unroll
        for (int t = 0; t < MT; t++) p.before[t] = KEEP || PAIR ? 0.f : held_output(out_at(t, 0), a.rows, accumulate && (uint32_t)t < a.m, lane < (uint32_t)OUTS, j);
        __builtin_amdgcn_sched_barrier(0);
    };
    Pass buf[2];
    fetch(first, buf[0]);
    // (KEEP: what the outputs of the lane's next store hold)
    float held[MT];
    auto ask_held = [&](uint32_t from) __attribute__((always_inline)) {
        const uint32_t j = (from + lane / OUTS * nwaves) * OUTS + lane % OUTS;
#pragma unroll
        for (int t = 0; t < MT; t++) held[t] = held_output(out_at(t, 0), a.rows, accumulate && (uint32_t)t < a.m, true, j);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (KEEP && !PAIR) ask_held(first);

    float scale[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) scale[t] = 1.0f;
    if (a.flags & FLAG_NORM) {
        float ss[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            ss[t] = 0.f;
#pragma unroll
            for (int j = 0; j < XV; j++)
                if (tid + 256u * j < k4) ss[t] += xv[t][j].x * xv[t][j].x + xv[t][j].y * xv[t][j].y + xv[t][j].z * xv[t][j].z + xv[t][j].w * xv[t][j].w;
            ss[t] = wave_sum(ss[t]);
        }
        if (lane == 0) {
#pragma unroll
            for (int t = 0; t < MT; t++) red[4 * t + wave] = ss[t];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const float total = (red[4 * t] + red[4 * t + 1]) + (red[4 * t + 2] + red[4 * t + 3]);
            scale[t] = 1.0f / sqrtf(total / (float)a.k + a.eps);
        }
    }
    // Even vectors first, the odd ones behind them: a task is two neighbouring vectors, and each
    // read below then covers consecutive ones.
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < XV; j++) {
            const uint32_t i = tid + 256u * j;
            if (i >= k4) continue;
            float4 v = xv[t][j];
            if (a.flags & FLAG_NORM) {
                v.x = v.x * scale[t] * gv[j].x; v.y = v.y * scale[t] * gv[j].y;
                v.z = v.z * scale[t] * gv[j].z; v.w = v.w * scale[t] * gv[j].w;
            }
            xs4[(uint32_t)t * k4 + (i & 1u) * (k4 / 2u) + (i >> 1)] = v;
        }
    __syncthreads();
    if (first >= passes) return;

    float x[MT][ITERS][8];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int it = 0; it < ITERS; it++) {
            const uint32_t task = lane + 64u * it;
            const bool mine = it < ITERS - 1 || task < tasks;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 v = xs4[(uint32_t)t * k4 + (uint32_t)h * (k4 / 2u) + (mine ? task : 0u)];
                // (a lane without a task multiplies zeros by zeros, whatever the inputs hold)
                x[t][it][4 * h] = mine ? v.x : 0.f; x[t][it][4 * h + 1] = mine ? v.y : 0.f;
                x[t][it][4 * h + 2] = mine ? v.z : 0.f; x[t][it][4 * h + 3] = mine ? v.w : 0.f;
            }
        }

    // Lane o < OUTS: its output's (gate) sum, and with PAIR the up row's; KEEP: those of the pass numbered turn are lanes turn OUTS + o.
    float v0[MT], v1[MT];
    uint32_t turn = 0, kept_first = first;
#pragma unroll
    for (int t = 0; t < MT; t++) v0[t] = v1[t] = 0.f;
    auto flush_kept = [&]() __attribute__((always_inline)) {
        const uint32_t j = (kept_first + lane / OUTS * nwaves) * OUTS + lane % OUTS;
        if (lane < turn * OUTS && j < a.rows) {
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if ((uint32_t)t >= a.m) break;
                float v = PAIR ? silu_f(v0[t]) * v1[t] : v0[t];
                float *o = out_at(t, j);
                if (accumulate) v += PAIR ? *o : held[t];
                *o = v;
            }
        }
        kept_first += turn * nwaves;
        turn = 0;
        if (!PAIR) ask_held(kept_first);
    };
    auto multiply = [&](uint32_t u, const Pass &p) __attribute__((always_inline)) {
        const uint32_t slot = KEEP ? turn * OUTS : 0u;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            float acc[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t] = 0.f;
#pragma unroll
            for (int it = 0; it < ITERS; it++) {
                float w[8];
                D::expand(make_uint4(p.q[r][it][0], p.q[r][it][1], p.q[r][it][2], p.q[r][it][3]), w);
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    float s = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; e++) s = fmaf(w[e], x[t][it][e], s);
                    acc[t] += s;
                }
            }
            constexpr int outs = OUTS;
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const float sum = wave_sum(acc[t]);
                if (PAIR && r >= outs) v1[t] = lane == slot + (uint32_t)(r - outs) ? sum : v1[t];
                else v0[t] = lane == slot + (uint32_t)r ? sum : v0[t];
            }
        }
        if (KEEP) {
            if (++turn == 64u / OUTS) flush_kept();
            return;
        }
        const uint32_t j = u * OUTS + lane;
        if (lane < (uint32_t)OUTS && j < a.rows) {
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if ((uint32_t)t >= a.m) break;
                float v = PAIR ? silu_f(v0[t]) * v1[t] : v0[t];
                if (accumulate) v += PAIR ? *out_at(t, j) : p.before[t];
                *out_at(t, j) = v;
            }
        }
    };
    for (uint32_t u = first;;) {
        fetch(u + nwaves, buf[1]);
        multiply(u, buf[0]);
        if ((u += nwaves) >= passes) break;
        fetch(u + nwaves, buf[0]);
        multiply(u, buf[1]);
        if ((u += nwaves) >= passes) break;
    }
    if (KEEP) flush_kept();
}

template <class D, int MT, int ITERS>
zhip_result launch_iters(const Dispatch &d, const MvArgs &a) {
    if (!MV_HOLDS(a)) return fail(d, ZHIP_E_GPU, "%s: k = %u", D::name(), a.k);
    // (Groups of tokens: blocks a multiple of the eight dies, so that the groups' workgroups of the same rows
    // share an L2; at three groups of 170 blocks 2 x 4096 x 2048 took 17.6 us instead of 12.4.)
    // Two workgroups a CU (three and more measured slower everywhere but on gate / up pairs of 200 MB:
    // 4096 x 4096 8.1, 8.7, 9.4 us at two, three, four a CU), a row a pass (a gate / up pair: its two rows),
    // two where a row is no more than two loads a lane: 2048 x 1024 2.9 -> 2.7 us, but 1024 x 2048 3.2 -> 3.4.
    const bool pair = (a.flags & FLAG_SILU_PAIR) != 0;
    constexpr int ROWS = ITERS <= 2 ? 2 : 1;
    const uint32_t outs = pair ? 1u : (uint32_t)ROWS;
    const uint32_t want = ((a.rows + outs - 1u) / outs + 3u) / 4u, groups = (a.m + MT - 1u) / MT, all = 2u * (uint32_t)d.dev->compute_units;
    uint32_t cap = all / groups, blocks = want < cap ? want : cap;
    if (groups > 1u) blocks = want < cap ? (want + 7u) & ~7u : cap & ~7u;
    const dim3 grid(blocks ? blocks : 1u, groups);
    const uint32_t lds = MT * a.k * 4u;
    // Stores between the loads of the stream cost more than their bytes: from the fourth pass of a wave on (a pair's from the sixth: 2 x 4096
    // x 2048 f16 at four tokens, four passes, 10.0 / 10.5 us, at eight, eight, 14.2 / 13.4) they wait in the lanes. us, stored pass by pass / kept, bf16: 151936 x 1024 at four / eight tokens 61.5 85.6 / 55.2 76.3, 50257 x 2560 61 88 / 57 76, 16384 x
    // 2048 15.4 23.1 / 14.0 20.2, 2 x 8192 x 2048 15.8 22.6 / 14.8 21.4, at one token level (151936 x 1024 52.1 / 51.9). Not a pair's
    // of longer rows, at any number of tokens: 2 x 9728 x 2560 at four 27.2 / 30.5 (at eight 36.1 / 32.6).
    constexpr bool PAIR_KEEPS = ITERS <= 4;
    const bool keep = (a.rows + outs - 1u) / outs > (pair ? 20u : 12u) * blocks;
    if constexpr (PAIR_KEEPS)
        if (pair && keep) {
            hipLaunchKernelGGL((matvec_half_row_kernel<D, MT, ITERS, true, 2, true>), grid, dim3(256), lds, d.stream, MV_GIVE_FIRST(MT, a, 0));
            return check_launch(d, D::name());
        }
    if (pair) hipLaunchKernelGGL((matvec_half_row_kernel<D, MT, ITERS, true, 2, false>), grid, dim3(256), lds, d.stream, MV_GIVE_FIRST(MT, a, 0));
    else if (keep) hipLaunchKernelGGL((matvec_half_row_kernel<D, MT, ITERS, false, ROWS, true>), grid, dim3(256), lds, d.stream, MV_GIVE_FIRST(MT, a, 0));
    else hipLaunchKernelGGL((matvec_half_row_kernel<D, MT, ITERS, false, ROWS, false>), grid, dim3(256), lds, d.stream, MV_GIVE_FIRST(MT, a, 0));
    return check_launch(d, D::name());
}

template <class D, int MT, int ITERS>
zhip_result launch_tokens(const Dispatch &d, const MvArgs &a) {
    if ((a.k + 511u) / 512u == (uint32_t)ITERS) return launch_iters<D, MT, ITERS>(d, a);
    if constexpr (ITERS > 1) return launch_tokens<D, MT, ITERS - 1>(d, a);
    return fail(d, ZHIP_E_BAD_COMMAND, "%s: k = %u", D::name(), a.k);
}

// The longest rows, in 512 weights, for a lane's inputs of one, two, up to four and up to eight tokens.
constexpr uint32_t kIters1 = 10, kIters2 = 6, kIters4 = 4, kIters8 = 2;

// How many tokens a workgroup takes: the fewer the sooner it has them in its registers and the more
// workgroups share the multiply, but each group of tokens reads the weights over again, from L2 where
// the groups keep step (their workgroups of the same rows lie on one die). us, tokens a workgroup in brackets:
//   five and eight tokens  2048 x 2048 (8 MB) 5.5 6.0 [2], 6.2 6.6 [4], 5.9 7.1 [1]; 2048 x 1024 3.9 4.1 [2], 4.6 5.0 [4], 6.0 6.2 [8]; 14336 x 1024 (29 MB) 12.1 12.7 [4], 13.0 13.2 [8],
//     40000 x 1024 (82 MB) 27.4 28.8 [4], 27.2 27.5 [8];
//     2 x 3072 x 1024 (13 MB) 7.6 8.5 [2], 7.6 8.7 [4], 9.2 10.4 [8]; 2 x 4096 x 2048 (34 MB) 12.4 14.5 [2], 12.9 13.9 [4];
//     14336 x 2048 (59 MB) 20.1 23.6 [2], 19.4 20.4 [4]; 151936 x 1024 at eight 128 [2], 101 [4], 86 [8]
//   three and four tokens  2048 x 2048 4.8 4.9 [2], 6.1 6.1 [4]; 2 x 3072 x 1024 5.8 6.0 [2], 6.1 6.8 [4]; 2 x 4096 x 2048 10.3 10.7
//     [2], 9.6 10.0 [4]; 32003 x 2048 (131 MB) 32.6 34.0 [2], 26.1 26.4 [4]
// and what ran matvec.hip's kernel before, for want of registers, now / then, at two, three, four and eight tokens:
//   2560 x 2560 at three, four, five and eight 6.2 6.4 6.8 7.8 [2] / 10.7 10.8 16.8 17.1; 32003 x 2560 (164 MB) at three, four and
//     eight 35.8 37.6 56.8 [2] / 42.6 43.7 75.0; 2048 x 2048 at five and eight 5.5 6.0 / 11.3 11.9
//   2560 x 3584 (18 MB) 7.0 7.5 8.2 11.6 [1] / 9.5 12.1 12.3 19.9; 4096 x 4096 (34 MB) 9.2 10.4 11.7 17.2 [1] / 11.5 13.5 13.6 22.7;
//     8192 x 4096 (67 MB) 15.5 17.5 20.3 31.0 [1] / 19.0 19.2 19.5 34.3, and past 60 MB it is that kernel's: 2 x 7168 x 3584
//     (103 MB) 30.9 30.8 33.0 46.7 / 24.2 24.2 24.6 43.9.
constexpr uint64_t kSplitBytes = 24ull << 20, kWideBytes = 40ull << 20, kLoneBytes = 60ull << 20;
uint64_t bytes_of(const MvArgs &a) { return (uint64_t)a.rows * a.row_bytes * ((a.flags & FLAG_SILU_PAIR) ? 2u : 1u); }

template <class D>
zhip_result launch(const Dispatch &d, const MvArgs &a) {
    const uint32_t iters = (a.k + 511u) / 512u;
    if (a.m == 1u || iters > kIters2) return launch_tokens<D, 1, kIters1>(d, a);
    if (a.m == 2u || iters > kIters4 || bytes_of(a) <= kSplitBytes) return launch_tokens<D, 2, kIters2>(d, a);
    if (a.m <= 4u || iters > kIters8 || bytes_of(a) <= kWideBytes) return launch_tokens<D, 4, kIters4>(d, a);
    return launch_tokens<D, 8, kIters8>(d, a);
}

}  // namespace

// The validated call of a 16-bit format: rows whose inputs of one token fit the registers, and a
// matrix (each half of a pair) that 32-bit offsets reach.
bool matvec_half_row_accepts(const MvArgs &a) {
    const uint32_t iters = (a.k + 511u) / 512u;
    return a.m <= 8u && iters <= kIters1 && (a.m == 1u || iters <= kIters2 || bytes_of(a) <= kLoneBytes) && (uint64_t)a.rows * a.row_bytes <= 0x7fffffffu;
}
zhip_result launch_matvec_half_row(const Dispatch &d, const MvArgs &a, bool f16) { return f16 ? launch<DecF16>(d, a) : launch<DecBF16>(d, a); }

}  // namespace zhip
