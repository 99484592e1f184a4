// Shared by the decode multiplies: their arguments and the input staging.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace zhip {

struct MvArgs {
    const float *x;
    const uint8_t *w;
    float *out;
    const float *norm_w;
    uint32_t n, k, col0, out_stride;
    float eps;
    uint32_t flags, half;
    uint32_t xr;         // floats between tokens' inputs
    uint32_t m;          // tokens
    uint32_t rows;       // outputs covered by the logical grid
    uint32_t row_bytes;  // bytes between weight rows
    float act_div;       // > 0: inputs staged as silu(x / act_div)
};

// What a multiply's first loads are addressed by comes ahead of its other parameters, as parameters of their own: the first fourteen
// words of those are in the wave's registers when it starts (the compiler's -amdgpu-kernarg-preload-count), a struct is
// fetched from memory first: 0.2 - 0.3 us of a launch (2 MB read by 256 workgroups 3.03 -> 2.82 us behind the launch before). us a
// token, 28 layers of 1024 x 3072 Q8_0 432 -> 391, bf16 486 -> 439; twelve of 2560 x 9728 Q5_K, two tokens, 513 -> 494. The outputs' stride gives its place to a gate / up step's `half`, and the count of tokens gives its to
// eps where a workgroup has one token: those are fetched behind the first loads, and late is soon enough for them. k and the flags
// share a word: rows of 16 M weights and more have no kernel that takes its parameters so, and each launch of one makes sure of it (MV_HOLDS).
#define MV_FIRST const float *first_x, const uint8_t *first_w, const float *first_norm_w, float *first_out, uint32_t first_k, uint32_t first_rows, \
    uint32_t first_row_bytes, uint32_t first_step, uint32_t first_xr, uint32_t first_m, float late_eps, float late_act_div, uint32_t late_out_stride
#define MV_TAKE_FIRST(MT, PAIR)                                                                                                                           \
    MvArgs { first_x, first_w, first_out, first_norm_w, 0u, first_k & 0xffffffu, 0u, PAIR ? late_out_stride : first_step,                                     \
        MT == 1 ? __uint_as_float(first_m) : late_eps, first_k >> 24, first_step, first_xr, MT == 1 ? 1u : first_m, first_rows, first_row_bytes, late_act_div }
// The tokens from t0 on.
#define MV_GIVE_FIRST(MT, a, t0) MV_GIVE_FIRST_AS(a, t0, MT == 1 ? __builtin_bit_cast(uint32_t, (a).eps) : (a).m - (t0))
#define MV_GIVE_FIRST_AS(a, t0, last) (a).x + (size_t)(t0) * (a).xr, (a).w, (a).norm_w, (a).out + (size_t)(t0) * (a).out_stride + (a).col0, (a).k | (a).flags << 24, (a).rows, \
    (a).row_bytes, (a).flags & FLAG_SILU_PAIR ? (a).half : (a).out_stride, (a).xr, last, (a).eps, (a).act_div, \
    (a).out_stride

// What shares a word keeps to its part of it.
#define MV_HOLDS(a) ((a).k < 1u << 24 && (a).flags < 1u << 8)

// What output j (below `rows`) of a token holds, for a step that adds to it: asked for with the rows it belongs to, since behind their
// sums it is one more trip to memory (us a token, 28 layers of 1024 x 3072 bf16 439 -> 422; eight of 4096 x 14336 Q4_K 379 -> 375). One load whatever the step and the lane, out of the buffer's range where there is nothing to add
// to: a load some waves leave out would have the others wait for one of the next rows' in its place.
__device__ __forceinline__ float held_output(const float *out, uint32_t rows, bool accumulate, bool mine, uint32_t j) {
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(out), 0, accumulate ? (int)(rows * 4u) : 0, 0x00020000);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, mine && j < rows ? 4u * j : 0x80000000u, 0, 0));
}

// The sum over a wave's lanes, in every lane: pairs 32, 16, 8, 4, 2 and 1 lanes apart, in that
// order. Nothing goes through LDS: the halves and the rows of sixteen trade places
// (v_permlane32_swap, v_permlane16_swap), the rest are DPP operands of the additions. A rotation
// by four reaches the lane four apart or the one four and eight apart, and after the step
// before those two hold the same sum. Six trips to LDS one after the other (ds_bpermute, what
// __shfl_xor compiles to) take about 0.3 us of a launch that lasts four.
template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    v = add_dpp<0x128>(v);  // row_ror:8
    v = add_dpp<0x124>(v);  // row_ror:4
    v = add_dpp<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    return add_dpp<0xB1>(v);  // quad_perm [1, 0, 3, 2]
}

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }

// Stages token `token`'s k inputs at dst (k / 4 vectors): normalised with the
// RMSNorm prologue and / or activated as silu(x / act_div) as the flags ask
// (src/kernels/matvec_quant.wgsl.hbs:73-89,175-198). Every thread of the
// 256-thread workgroup must call it; `red` is four floats of LDS. Vector i of
// the token lands at dst[place(i)].
template <class Place>
__device__ __forceinline__ void stage_token(const MvArgs &a, uint32_t token, float4 *dst, float *red, Place place) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t k4 = a.k / 4u;
    const float4 *xrow = reinterpret_cast<const float4 *>(a.x + (size_t)token * a.xr);
    float scale = 1.0f;
    if (a.flags & FLAG_NORM) {
        float ss = 0.f;
        for (uint32_t i = tid; i < k4; i += 256u) {
            const float4 v = xrow[i];
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
        ss = wave_sum(ss);
        __syncthreads();
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        ss = (red[0] + red[1]) + (red[2] + red[3]);
        scale = 1.0f / sqrtf(ss / (float)a.k + a.eps);
    }
    const float4 *nw = reinterpret_cast<const float4 *>(a.norm_w);
    for (uint32_t i = tid; i < k4; i += 256u) {
        float4 v = xrow[i];
        if (a.flags & FLAG_NORM) {
            const float4 g = nw[i];
            v.x = v.x * scale * g.x; v.y = v.y * scale * g.y;
            v.z = v.z * scale * g.z; v.w = v.w * scale * g.w;
        }
        if (a.act_div > 0.f) {
            v.x = silu_f(v.x / a.act_div); v.y = silu_f(v.y / a.act_div);
            v.z = silu_f(v.z / a.act_div); v.w = silu_f(v.w / a.act_div);
        }
        dst[place(i)] = v;
    }
}

__device__ __forceinline__ void stage_token(const MvArgs &a, uint32_t token, float4 *dst, float *red) {
    stage_token(a, token, dst, red, [](uint32_t i) { return i; });
}

// Matrix-core variants over rows of more than 4096 weights: `parts` workgroups share a tile, each
// over 2048 of its columns, and leave their sums in `partial` ([part][gate, up][token of 8][output],
// outputs a.rows apart); this launch adds a tile's parts in the order of their columns and applies
// the SILU_PAIR / ACCUMULATE epilogue (matvec_mfma_resident.hip).
constexpr uint32_t kMatvecMaxParts = 16;  // rows of up to 32768 weights
// The 16-bit matrices of whole 512s a row that ZHIP_OPTION_WIDE_DECODE moves to the matrix cores (matvec.hip).
constexpr uint64_t kMatvecBf16StreamBytes = 16ull << 20;
zhip_result launch_matvec_parts_sum(const Dispatch &d, const char *name, const MvArgs &a, const float *partial, uint32_t parts);
// A step over such rows with the RMSNorm prologue: no workgroup sees a whole row, so a launch of
// its own leaves each token's 1 / sqrt(mean(x^2) + eps) in scales[token] beforehand (the sum of
// squares as stage_token takes it). The workspace's first kPartsScalesBytes hold them.
constexpr uint32_t kPartsScalesBytes = 64;
zhip_result launch_matvec_parts_scales(const Dispatch &d, const char *name, const MvArgs &a, float *scales);

}  // namespace zhip
