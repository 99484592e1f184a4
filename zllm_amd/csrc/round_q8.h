// How quantize_q8 rounds a 32-value block (llama.cpp's Q8_0 activations, src/ref/matmul.zig:197-247): eight lanes, four values each.
// Every operation whose rounding decides a value is an operation of its own, so that the compiler can neither fuse nor approximate it.
#pragma once

#include <hip/hip_runtime.h>

namespace zhip {

typedef float qf32x4 __attribute__((ext_vector_type(4)));

// ggml's nearest_int: adding 1.5 * 2^23 rounds the f32 to an integer, ties to even.
__device__ __forceinline__ int nearest_int(float y) {
    return __float_as_int(__fadd_rn(y, 12582912.0f)) - 0x4b400000;
}

// max over lane pairs, quads and groups of eight: every lane of the group ends with the group's maximum.
template <int CTRL>
__device__ __forceinline__ float max_with(float v) {
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float max_of_eight(float v) {
    v = max_with<0xB1>(v);   // quad_perm [1, 0, 3, 2]
    v = max_with<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    return max_with<0x141>(v);  // row_half_mirror: the other quad of the eight
}

// The lane's four 8-bit values of its block, whose largest magnitude is amax, and the block's scale.
__device__ __forceinline__ float round_block(const qf32x4 &v, float amax, int (&q)[4]) {
#pragma unroll
    for (int e = 0; e < 4; e++) q[e] = 0;
    if (amax == 0.f) return 0.f;
    const float d32 = __fdiv_rn(amax, 127.0f);
    const float id = __fdiv_rn(127.0f, amax);
#pragma unroll
    for (int e = 0; e < 4; e++) q[e] = nearest_int(__fmul_rn(v[e], id));
    return (float)(_Float16)d32;
}
__device__ __forceinline__ uint32_t four_bytes(const int (&q)[4]) {
    return ((uint32_t)q[0] & 0xffu) | (((uint32_t)q[1] & 0xffu) << 8) | (((uint32_t)q[2] & 0xffu) << 16) | (((uint32_t)q[3] & 0xffu) << 24);
}

// silu(gate) * up (src/kernels/silu_mul.wgsl), four values.
__device__ __forceinline__ qf32x4 silu_pair(const qf32x4 &gate, const qf32x4 &up) {
    qf32x4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = gate[i] / (1.0f + expf(-gate[i])) * up[i];
    return v;
}

}  // namespace zhip
