// quantize_q8: rows of activations rounded to 8-bit blocks for the int8 prefill
// multiply, value for value as llama.cpp's x86 CPU backend rounds them
// (src/kernels/quantize_q8.wgsl, src/ref/matmul.zig:197-247). A wave takes a
// chunk of 256 values of a row, four values a lane
// (a chunk is one Q8_K block, or eight Q8_0 blocks of eight lanes each), and a
// workgroup is four such waves on neighbouring chunks. A chunk's rounding is a
// chain of dependent operations behind one 16-byte load, so what hides it is
// other waves. With the RMSNorm prologue every workgroup of a row (one to eight: see
// launch_norm) first adds the whole row's squares together and then rounds its share of the chunks. The largest magnitude of a
// block is found with row-local DPP steps (and, for Q8_K, four lane reads),
// the first position that holds it with a ballot. Every operation whose rounding
// decides a value is an operation of its own (the library is compiled with
// -ffp-contract=on, which fuses only within one source expression, and with
// hipcc's correctly rounded f32 division and square root), so the compiler can
// neither fuse the multiply into the rounding addition nor approximate a division.
#include <hip/hip_runtime.h>

#include "common.h"
#include "round_q8.h"

namespace zhip {

struct QuantizeQ8Params {  // params.QuantizeQ8 (src/kernels/kernels.zig:495-501)
    uint32_t k, block, mode;
    float eps;
};
static_assert(sizeof(QuantizeQ8Params) == 16, "params.QuantizeQ8 is 16 bytes");

// The same over a wave.
__device__ __forceinline__ float max_of_wave(float v) {
    v = max_with<0x140>(max_of_eight(v));  // row_mirror: the other eight of the row
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)), b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32)), d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// The 8-bit values of one 256-value chunk of a row, four a lane from `first` on (lanes past the row hold zeros and
// store nothing), and its scale or scales.
__device__ __forceinline__ void round_chunk(const QuantizeQ8Params &p, const qf32x4 &v, bool live, size_t base, uint32_t lane, uint32_t *qx, float *dx) {
    // The lane's first largest magnitude: a strict > scan from the left.
    float mag = fabsf(v[0]), value = v[0];
#pragma unroll
    for (int e = 1; e < 4; e++) {
        const float a = fabsf(v[e]);
        if (a > mag) {
            mag = a;
            value = v[e];
        }
    }
    int q[4] = {0, 0, 0, 0};
    float d = 0.f;
    if (p.block == 256u) {
        // Q8_K: the value itself (with its sign) at the first position of the largest
        // magnitude: the lowest lane that holds it.
        const float amax = max_of_wave(mag);
        const uint64_t holders = __ballot(mag == amax);
        const float lead = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(value), (int)__ffsll((unsigned long long)holders) - 1));
        if (amax != 0.f) {
            const float iscale = __fdiv_rn(-127.0f, lead);
            d = __fdiv_rn(1.0f, iscale);
#pragma unroll
            for (int e = 0; e < 4; e++) q[e] = min(127, nearest_int(__fmul_rn(iscale, v[e])));
        }
    } else {
        d = round_block(v, max_of_eight(mag), q);
    }
    if (!live) return;
    qx[base / 4u] = four_bytes(q);
    if (((4u * lane) & (p.block - 1u)) == 0u) dx[base >> (p.block == 256u ? 8 : 5)] = d;  // (a division by the block would be one of 64 bits)
}

// A double of each lane plus that of the lane 32, 16, 8, 4, 2 and 1 away (by turns: after the step of 8 the rows
// of sixteen repeat every eight lanes, so a rotation by 4 is the exchange): every lane ends with the wave's sum.
template <int CTRL>
__device__ __forceinline__ double add_with(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, true), hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double sum_of_wave(double v) {
    uint64_t b = __builtin_bit_cast(uint64_t, v);
    const auto lo32 = __builtin_amdgcn_permlane32_swap((uint32_t)b, (uint32_t)b, false, false), hi32 = __builtin_amdgcn_permlane32_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    v = __builtin_bit_cast(double, (uint64_t)hi32[0] << 32 | lo32[0]) + __builtin_bit_cast(double, (uint64_t)hi32[1] << 32 | lo32[1]);
    b = __builtin_bit_cast(uint64_t, v);
    const auto lo16 = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false), hi16 = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    v = __builtin_bit_cast(double, (uint64_t)hi16[0] << 32 | lo16[0]) + __builtin_bit_cast(double, (uint64_t)hi16[1] << 32 | lo16[1]);
    v = add_with<0x128>(v);     // row_ror:8
    v = add_with<0x124>(v);     // row_ror:4
    v = add_with<0x4E>(v);      // quad_perm [2, 3, 0, 1]
    return add_with<0xB1>(v);   // quad_perm [1, 0, 3, 2]
}
// The RMSNorm factor as ggml computes it (src/ref/ops.zig:25-41): f32 squares
// summed and divided in f64, an f32 mean, add, sqrt and reciprocal (then x * scale, then * w).
__device__ __forceinline__ float norm_factor(const QuantizeQ8Params &p, double ss, double (&squares)[4]) {
    ss = sum_of_wave(ss);
    if ((threadIdx.x & 63u) == 0u) squares[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = (squares[0] + squares[1]) + (squares[2] + squares[3]);
    const float mean = (float)(ss / (double)p.k);
    // (sqrtf is the correctly rounded square root under hipcc's default options; the
    // __fsqrt_rn intrinsic is the hardware's approximate one here and gave some rows a
    // scale one unit in the last place away from ggml's)
    return __fdiv_rn(1.0f, sqrtf(__fadd_rn(mean, p.eps)));
}

// The RMSNorm prologue over a row of up to 1024 J values: the row and its weights are read once and
// kept in registers. gridDim.x workgroups a row: each adds up the whole row's squares and rounds its share of the
// chunks. What bounds it is the chain of the two trips (the row, the stores) and a wave's rounding, 0.2 us a chunk
// where it has the SIMD to itself. us, a row read twice by one workgroup (once for the sum) / this: 64 x 4096 4.6 / 2.5, 64 x 5120
// 6.2 / 2.9, 128 x 4096 4.6 / 2.8, 201 x 2560 4.4 / 3.1, 512 x 1024 3.1 / 2.4, 512 x 4096 6.0 / 4.8.
template <int J>
__global__ __launch_bounds__(256) void quantize_q8_norm_kernel(const float *x, uint32_t *qx, float *dx, const float *nw, uint32_t k, uint32_t block, uint32_t mode, float eps) {
    const QuantizeQ8Params p{k, block, mode, eps};
    __shared__ double squares[4];
    const uint32_t at = 4u * threadIdx.x;
    const size_t row = (size_t)blockIdx.y * p.k;
    qf32x4 v[J], w[J];
#pragma unroll
    for (int j = 0; j < J; j++) v[j] = at + 1024u * j < p.k ? *reinterpret_cast<const qf32x4 *>(x + row + at + 1024u * j) : qf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; j++) w[j] = *reinterpret_cast<const qf32x4 *>(nw + (at + 1024u * j < p.k ? at + 1024u * j : 0u));
    double ss = 0.0;
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) ss += (double)__fmul_rn(v[j][e], v[j][e]);
    const float scale = norm_factor(p, ss, squares);
#pragma unroll
    for (int j = 0; j < J; j++) {
        if (J > 1 && j % gridDim.x != blockIdx.x) continue;
        const bool live = at + 1024u * j < p.k;
#pragma unroll
        for (int e = 0; e < 4; e++) v[j][e] = live ? __fmul_rn(__fmul_rn(v[j][e], scale), w[j][e]) : 0.f;
        round_chunk(p, v[j], live, row + at + 1024u * j, threadIdx.x & 63u, qx, dx);
    }
}
// The same over rows of any length, read twice.
__global__ __launch_bounds__(256) void quantize_q8_norm_long_kernel(const float *x, uint32_t *qx, float *dx, const float *nw, uint32_t k, uint32_t block, uint32_t mode, float eps) {
    const QuantizeQ8Params p{k, block, mode, eps};
    __shared__ double squares[4];
    const uint32_t at = 4u * threadIdx.x;
    const size_t row = (size_t)blockIdx.y * p.k;
    auto four = [&](const float *from, uint32_t i0, qf32x4 (&r)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) r[j] = i0 + 1024u * j < p.k ? *reinterpret_cast<const qf32x4 *>(from + i0 + 1024u * j) : qf32x4{0.f, 0.f, 0.f, 0.f};
    };
    double ss = 0.0;
    for (uint32_t i0 = at; i0 < p.k; i0 += 4096u) {
        qf32x4 r[4];
        four(x + row, i0, r);
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) ss += (double)__fmul_rn(r[j][e], r[j][e]);
    }
    const float scale = norm_factor(p, ss, squares);
    for (uint32_t i0 = at; i0 - at < p.k; i0 += 4096u) {  // (whole waves: a chunk's lanes look at each other)
        qf32x4 r[4], w[4];
        four(x + row, i0, r);
        four(nw, i0, w);
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const bool live = i0 + 1024u * j < p.k;
#pragma unroll
            for (int e = 0; e < 4; e++) r[j][e] = live ? __fmul_rn(__fmul_rn(r[j][e], scale), w[j][e]) : 0.f;
            round_chunk(p, r[j], live, row + i0 + 1024u * j, threadIdx.x & 63u, qx, dx);
        }
    }
}

// Without the prologue: a chunk a wave.
__global__ __launch_bounds__(256) void quantize_q8_kernel(const float *x, uint32_t *qx, float *dx, uint32_t k, uint32_t block, uint32_t mode) {
    const QuantizeQ8Params p{k, block, mode, 0.f};
    const uint32_t at = 1024u * blockIdx.x + 4u * threadIdx.x;
    const bool live = at < p.k;
    const size_t row = blockIdx.y;
    qf32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (p.mode == 2u) {
        // silu(gate) * up over a row of gate | up (src/kernels/silu_mul.wgsl).
        const float *g = x + row * 2u * p.k + (live ? at : 0u);
        qf32x4 gate = *reinterpret_cast<const qf32x4 *>(g), up = *reinterpret_cast<const qf32x4 *>(g + p.k);
        // (zeros give zeros: no branch around each of the four, whose chains overlap)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            gate[i] = live ? gate[i] : 0.f;
            up[i] = live ? up[i] : 0.f;
        }
        v = silu_pair(gate, up);
    } else if (live) {
        v = *reinterpret_cast<const qf32x4 *>(x + row * p.k + at);
    }
    round_chunk(p, v, live, row * p.k + at, threadIdx.x & 63u, qx, dx);
}

// Workgroups a row: as many as leave each a CU of its own, two up to a row a CU. One / two / four (0.25 us ahead
// of the kernel as it is): 64 x 4096 4.1 / 3.2 / 2.7 us, 128 x 4096 4.2 / 3.3 / 3.5, 201 x 2560 3.5 / 3.4 / 3.4, 256 x 1792 3.0 / 2.6,
// 256 x 4096 4.2 / 4.3 / 6.2; past it 300 x 5120 5.8 / 6.8 / 7.7, 512 x 2048 3.2 / 4.0, 512 x 4096 5.6 / 6.9 / 9.3.
template <int J>
static void launch_norm(const Dispatch &d, const QuantizeQ8Params &p, uint32_t spans, const float *x, uint32_t *qx, float *dx, const float *nw) {
    if constexpr (J < 8) {
        if (spans > (uint32_t)J) return launch_norm<J + 1>(d, p, spans, x, qx, dx, nw);
    }
    const uint32_t rows = d.grid[1], cus = (uint32_t)d.dev->compute_units;
    const uint32_t each = cus / rows > 2u ? cus / rows : 2u, parts = rows > cus ? 1u : each < (uint32_t)J ? each : (uint32_t)J;
    hipLaunchKernelGGL(quantize_q8_norm_kernel<J>, dim3(parts, rows), dim3(256), 0, d.stream, x, qx, dx, nw, p.k, p.block, p.mode, p.eps);
}

zhip_result launch_quantize_q8(const Dispatch &d) {
    if (d.params_size < sizeof(QuantizeQ8Params)) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: params block too small");
    const QuantizeQ8Params &p = *reinterpret_cast<const QuantizeQ8Params *>(d.params);
    for (int b = 1; b <= 4; b++)
        if (!d.bind[b].bound) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: binding %d is not bound", b);
    if (d.grid[0] == 0 || d.grid[1] == 0 || d.grid[2] == 0) return ZHIP_OK;
    if (d.grid[2] != 1) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: grid z must be 1");
    if (p.block != 32u && p.block != 256u) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: block = %u (32 or 256)", p.block);
    if (p.k == 0 || p.k % p.block != 0) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: k = %u is not a multiple of the block %u", p.k, p.block);
    if (p.mode > 2u) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: mode = %u", p.mode);
    const uint64_t chunks = (p.k + 255u) / 256u;
    if (d.grid[0] != chunks) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: grid x = %u, k = %u needs %llu", d.grid[0], p.k, (unsigned long long)chunks);
    if (d.grid[1] > 65535u) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: more than 65535 rows in one dispatch");
    const uint64_t rows = d.grid[1];
    const uint64_t x_need = rows * p.k * (p.mode == 2u ? 8u : 4u);
    const uint64_t q_need = rows * p.k, d_need = rows * (p.k / p.block) * 4u;
    if (x_need > d.bind[1].size || q_need > d.bind[2].size || d_need > d.bind[3].size || (p.mode == 1u && (uint64_t)p.k * 4u > d.bind[4].size))
        return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: bound ranges too small");
    if (((uintptr_t)d.bind[1].ptr | (p.mode == 1u ? (uintptr_t)d.bind[4].ptr : 0)) & 15u) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: x and norm weights must be 16-byte aligned");
    if (((uintptr_t)d.bind[2].ptr | (uintptr_t)d.bind[3].ptr) & 3u) return fail(d, ZHIP_E_BAD_COMMAND, "quantize_q8: outputs must be 4-byte aligned");
    if (d.rounds) {
        if (p.block == 32u) *d.rounds = RoundedCopy{reinterpret_cast<const float *>(d.bind[1].ptr), (uint32_t)rows, p.k, p.mode, d.bind[2].ptr, d.bind[3].ptr, nullptr, nullptr};
        return ZHIP_OK;
    }
    const float *x = reinterpret_cast<const float *>(d.bind[1].ptr), *nw = reinterpret_cast<const float *>(d.bind[4].ptr);
    uint32_t *qx = reinterpret_cast<uint32_t *>(d.bind[2].ptr);
    float *dx = reinterpret_cast<float *>(d.bind[3].ptr);
    // One chunk a wave, whatever the size: against two and four, inputs in the Infinity Cache, 512 x 3072 with the
    // SiLU-pair prologue 4.7 / 5.5 / 6.3 us, 512 x 4096 without one 3.8 / 3.9 / 4.2, 512 x 14336 with the prologue
    // 13.9 / 13.8 / 15.9, 201 x 9728 with it 5.3 / 5.9 / 7.5; only 512 x 14336 without one is faster with
    // two, 8.9 / 8.6. (With the block's index shifted, not divided: 4.5, -, 13.1 and 5.5 us.)
    const uint32_t spans = (d.grid[0] + 3u) / 4u;
    if (p.mode != 1u) hipLaunchKernelGGL(quantize_q8_kernel, dim3(spans, d.grid[1]), dim3(256), 0, d.stream, x, qx, dx, p.k, p.block, p.mode);
    else if (spans <= 8u) launch_norm<1>(d, p, spans, x, qx, dx, nw);
    else hipLaunchKernelGGL(quantize_q8_norm_long_kernel, dim3(1, d.grid[1]), dim3(256), 0, d.stream, x, qx, dx, nw, p.k, p.block, p.mode, p.eps);
    return check_launch(d, "quantize_q8");
}

}  // namespace zhip
