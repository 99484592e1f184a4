// matvec_q3_k / matvec_q4_k / matvec_q5_k / matvec_q6_k / matvec_q8_0, matrix-core variant (MatvecVariant wg 512, lanes 64, rows 16) for
// rows of any length and steps of up to eight tokens. Contract as the other variants
// (src/kernels/matvec_quant.wgsl.hbs); a token's result does not depend on how many tokens share
// the launch.
//
// Arithmetic. v_mfma_f32_16x16x32_f16 multiplies sixteen operand rows (a token is two: the f16 rounding of
// its inputs and that of what the rounding left, 22 bits, under a power of two a token and 256-weight
// block) by sixteen matrix rows over a 32-weight unit. The K formats' weights enter with their integer scale multiplied in,
// exact in f16 (s * q has up to 11 bits; Q6_K's 13 are two values), so that a block's units
// add up in the instruction's f32 accumulators (two or four of them: shorter sums) and d, dmin and the token's power of two are applied once a
// block; the minimums are an instruction of the units' input sums. Q8_0's scale, eleven bits of its own,
// is applied to a unit's sum.
//
// Layout. A workgroup of sixteen waves takes tiles of sixteen rows (eight where whole tiles do not
// share out), all of k: a wave has one or two (Q6_K: one) blocks of every row of its tiles, and of rows of up to half
// (a quarter) as many blocks as waves two (four) teams take a tile each. The wave brings its blocks' inputs
// in, turns them into operands through its own LDS and keeps them in registers; its weights arrive by direct loads of
// 16 bytes a lane, sixteen rows' pieces in a row, two or one blocks ahead in slots of its own: it waits
// for no one. One barrier a round, behind which two waves add the partial sums of a tile and
// store. The RMSNorm factor is left to the outputs, so nothing waits for the row's squares either. Rows of more than
// 8192 weights (Q6_K: 4096) are shared by k / 4096 workgroups, which leave their sums to a launch of their own.
//
// What bounds it: short launches the chain launch - inputs - operands - multiply - sum, of which the
// operands' VALU and LDS work grows with the tokens (0.3 us a token at k = 4096, every workgroup the
// same); long ones vector issue (Q4_K 158 vector instructions a block, Q6_K about 330) beside HBM.
// Scalar instructions count, sixteen waves sharing one scalar unit: a token's buffer each instead of one for all of
// them, runtime team counts and sums held over two rounds cost 0.5 us a launch. Eight waves a workgroup with twice
// the blocks each were slower (Q4_K 4096 x 4096 at four tokens 8.8 against 7.6 us), and so were parts of eight blocks
// (4096 x 14336 16.0 against 14.4). Measured against the kernels before (us at one / four / eight tokens, weights from HBM, with RMSNorm but for
// 4096 x 14336): Q4_K 4096 x 4096 10.3 10.3 10.8 -> 6.9 7.6 10.0, Q6_K 14.8 14.7 15.5 -> 7.9 8.3 10.1, Q3_K 12.8 12.7 13.3 -> 6.7 7.4 9.4,
// Q8_0 10.9 10.9 11.3 -> 7.8 8.1 9.9, Q4_K 2 x 14336 x 4096 21.7 21.2 21.8 -> 19.7 19.5 21.4, Q5_K 27.5 27.7 28.3 -> 22.4 22.0 24.5, Q6_K 4096 x 14336
// 19.9 19.9 20.7 -> 17.9 18.1 20.0; lengths that ran the default variant before: Q4_K 4096 x 2560 5.1 9.2 18.0 -> 6.3 7.1 9.6, Q5_K
// 2 x 9728 x 2560 12.3 28.7 57.0 -> 16.8 17.4 19.9, Q4_K 2560 x 9728 8.2 17.8 33.0 -> 10.2 10.8 12.9, Q8_0 2 x 9728 x 2560
// 12.0 25.4 49.9 -> 16.2 16.7 19.0 (one and two tokens pay for it, as on every matrix under this id). Where eight tokens pay too, matvec.hip says so.
//
// Precision. Those lengths had f32 inputs in the default variant; here an input has 22 bits and its sign, 23 in all, down to 2^-17 of its block's largest
// and fewer below (what is lost there is under 2^-39 of that largest). The outputs are the nearer ones to the exact all the same, since the sums are
// shorter (relative error against float64, 48 tokens over rows of 1280 .. 6912 weights, default / here): Q8_0 1.22 - 1.29e-7 / 0.86 - 0.96e-7, Q3_K 1.95 - 2.00e-7 / 0.87 -
// 0.96e-7, Q4_K 1.27 - 1.30e-7 / 1.03 - 1.11e-7, Q5_K 1.29 - 1.31e-7 / 1.07 - 1.12e-7, Q6_K 2.11 - 2.13e-7 / 1.00 - 1.08e-7, with RMSNorm 1.37 - 2.22e-7 / 1.06 - 1.31e-7; with
// every 256th input a thousand times the others 1.44 - 3.34e-7 / 1.04 - 1.59e-7.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "decode.h"
#include "matvec_common.h"

namespace zhip {

namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr;

constexpr uint32_t WAVES = 16, THREADS = 64 * WAVES;
// The operands of four tokens and a 256-weight block, in the wave's own LDS: eight 32-weight units of four
// groups of eight positions, each eight operand rows of 16 bytes and 16 bytes of padding; then the
// inverses of the tokens' scales and the eight rows' unit sums.
constexpr uint32_t GROUP = 8u * 16u + 16u, INVERSE_AT = 32u * GROUP, SUMS_AT = INVERSE_AT + 16u, OPERANDS = SUMS_AT + 128u;

constexpr uint32_t kMaxParts = 8;  // rows of up to 32768 weights
constexpr uint32_t kOutBytes = 0x7fffffff;  // how far behind a.out a step that accumulates reads
constexpr uint32_t kScales = kMaxParts * 8u, kSums = kScales + 8u;

struct RowsArgs {
    MvArgs a;
    uint32_t blocks;               // of 256 weights a row, the last one possibly short
    uint32_t groups;               // workgroups
    uint32_t rounds, left, split;  // (see the kernel's tiles)
    uint32_t parts;                // workgroups that share a tile, each over some of its blocks,
    float *partial;                // and where: [part][token of 8] sums of squares,
                                   // each token's norm factor where it goes through the activation, [part][gate, up][token of 8][output]
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buffer(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void load_lds_b128(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t offset, uint32_t uniform_offset) {
    asm volatile("" : "+s"(dst));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)dst, 16, offset, uniform_offset, 0, 0);
}
__device__ __forceinline__ void load_lds_b32(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t offset) {
    asm volatile("" : "+s"(dst));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)dst, 4, offset, 0, 0, 0);
}
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
template <int LEFT>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}
// A 4-byte store the compiler's wait-count bookkeeping does not see as a store: with one
// pending it would turn every wait for a load into a wait for all loads in flight.
__device__ __forceinline__ void store_apart(float *at, float v) {
    asm volatile("global_store_dword %0, %1, off\n\ts_nop 0" ::"v"(at), "v"(v) : "memory");
}
template <int CTRL>
__device__ __forceinline__ float from_dpp(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true)); }
// Each of G = 2 or 4 tokens' values put together over the wave: token lane % G's, in every lane. (Neighbours
// first trade tokens, so that the rest is one chain; the same pairs whichever G.)
template <int G, class Op>
__device__ __forceinline__ float over_tokens(const float (&v)[G], uint32_t lane, Op op) {
    float r[G / 2];
#pragma unroll
    for (int i = 0; i < G / 2; i++) {
        const float keep = (lane & 1u) ? v[2 * i + 1] : v[2 * i], give = (lane & 1u) ? v[2 * i] : v[2 * i + 1];
        r[i] = op(keep, from_dpp<0xB1>(give));
    }
    if constexpr (G == 4) {
        const float keep = (lane & 2u) ? r[1] : r[0], give = (lane & 2u) ? r[0] : r[1];
        r[0] = op(keep, from_dpp<0x4E>(give));
    } else {
        r[0] = op(r[0], from_dpp<0x4E>(r[0]));
    }
    r[0] = op(r[0], from_dpp<0x124>(r[0]));  // row_ror:4
    r[0] = op(r[0], from_dpp<0x128>(r[0]));  // row_ror:8
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(r[0]), __float_as_uint(r[0]), false, false);
    r[0] = op(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(r[0]), __float_as_uint(r[0]), false, false);
    return op(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
}

__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits) { return (v & mask) | bits; }
__device__ __forceinline__ f16x2 as_f16(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ f16x8 pack(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return __builtin_bit_cast(f16x8, u32x4{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)});
}
__device__ __forceinline__ f16x2 fma2(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ f32x4 mfma(f16x8 tokens, f16x8 weights, f32x4 sum) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(tokens, weights, sum, 0, 0, 0); }

// Q4_K and Q5_K: a weight is d * (s * q) - dmin * m with s, m 6 bits; s * q is exact in f16, and the
// minimums' part is a matrix instruction of the units' input sums against the eight m.
template <bool FIFTH>
struct RowsQ45 {
    static constexpr uint32_t BLOCK = FIFTH ? 176 : 144, CHUNKS = BLOCK / 16;
    static constexpr uint32_t SLOTS = 3;
    static constexpr uint32_t MOST = 2;   // blocks a wave keeps of a row
    static constexpr bool MINS = true;    // has minimums
    static constexpr bool RAGGED = false;  // rows are whole blocks
    static constexpr bool SPLIT = false;   // a row's scales lie behind its weights
    static constexpr uint32_t TYPE = FIFTH ? 5 : 4;
    static const char *name() { return FIFTH ? "matvec_q5_k" : "matvec_q4_k"; }
    // 16-byte chunk c of block b of a row of k weights, as bytes from the row's start.
    static __device__ __forceinline__ uint32_t chunk_at(uint32_t, uint32_t b, uint32_t c, uint32_t) { return BLOCK * b + 16u * c; }
    // Adds the block's products with the tokens' operands to out (operand rows 4 g .. + 3 of the lane's matrix row).
    static __device__ __forceinline__ void multiply(const uint8_t *slot, uint32_t l16, uint32_t g, uint32_t, const f16x8 (&xf)[8], const f16x8 &xsum, const float (&inv)[2], f32x4 &out) {
        const uint8_t *row = slot + BLOCK * l16;
        const u32x4 h = *reinterpret_cast<const u32x4 *>(row);
        const float d = half_bits_to_float(h.x & 0xffffu), dmin = half_bits_to_float(h.x >> 16);
        const uint32_t sc[2] = {h.y & 0x3f3f3f3fu, (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u)};
        const uint32_t mn[2] = {h.z & 0x3f3f3f3fu, ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u)};
        u32x2 fifth = {0u, 0u};
        if (FIFTH) fifth = *reinterpret_cast<const u32x2 *>(row + 16u + 8u * g);
        f32x4 sums[2] = {};  // of the chunks' low and high nibbles: shorter sums
        f16x2 m[4];
        const f16x2 minus = {(_Float16)-1024.f, (_Float16)-1024.f};
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            const u32x2 w = *reinterpret_cast<const u32x2 *>(row + BLOCK - 128u + 32u * c + 8u * g);
            // The chunk's two scales and minimums as f16: 1024 + value in the mantissa, less 1024.
            const uint32_t sel = (c & 1u) ? 0x04030402u : 0x04010400u;
            const f16x2 s = as_f16(__builtin_amdgcn_perm(0x64u, sc[c >> 1], sel)) + minus;
            m[c] = as_f16(__builtin_amdgcn_perm(0x64u, mn[c >> 1], sel)) + minus;
            const f16x2 off = s * f16x2{(_Float16)-1024.f, (_Float16)-64.f};
            const f16x2 s0 = {s[0], s[0]}, s1 = {s[1], s[1]}, o0 = {off[0], off[0]}, o1 = {off[1], off[1]};
            const uint32_t x8 = w.x >> 8, y8 = w.y >> 8;
            // Low nibbles under the exponent of 1024, high ones, four bits up, under that of 64.
            uint32_t lo[4] = {and_or(w.x, 0x000f000fu, 0x64006400u), and_or(x8, 0x000f000fu, 0x64006400u), and_or(w.y, 0x000f000fu, 0x64006400u), and_or(y8, 0x000f000fu, 0x64006400u)};
            uint32_t hi[4] = {and_or(w.x, 0x00f000f0u, 0x54005400u), and_or(x8, 0x00f000f0u, 0x54005400u), and_or(w.y, 0x00f000f0u, 0x54005400u), and_or(y8, 0x00f000f0u, 0x54005400u)};
            if (FIFTH) {  // bit 2 c (2 c + 1) of a position's byte above its nibble
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t f = e < 2 ? fifth.x : fifth.y;
                    const int at = 8 * (e & 1);
                    const int down0 = (int)(2u * c) + at - 4, down1 = (int)(2u * c + 1u) + at - 8;
                    lo[e] |= (down0 >= 0 ? f >> (down0 & 31) : f << (-down0 & 31)) & 0x00100010u;
                    hi[e] |= (down1 >= 0 ? f >> (down1 & 31) : f << (-down1 & 31)) & 0x01000100u;
                }
            }
            sums[0] = mfma(xf[2 * c], pack(fma2(as_f16(lo[0]), s0, o0), fma2(as_f16(lo[1]), s0, o0), fma2(as_f16(lo[2]), s0, o0), fma2(as_f16(lo[3]), s0, o0)), sums[0]);
            sums[1] = mfma(xf[2 * c + 1], pack(fma2(as_f16(hi[0]), s1, o1), fma2(as_f16(hi[1]), s1, o1), fma2(as_f16(hi[2]), s1, o1), fma2(as_f16(hi[3]), s1, o1)), sums[1]);
        }
        const f32x4 mins = mfma(xsum, pack(m[0], m[1], m[2], m[3]), f32x4{0.f, 0.f, 0.f, 0.f});
        const float less = -32.f * dmin;
#pragma unroll
        for (int e = 0; e < 4; e++) out[e] = fmaf(inv[e >> 1], fmaf(d, sums[0][e] + sums[1][e], less * mins[e]), out[e]);
    }
};

// Q6_K (blocks padded to 224 bytes): a weight is d * s * (q - 32) with s a signed byte for sixteen weights. The
// product s * (q - 32) has up to 13 bits: its rounding to f16 and what that leaves are an instruction each.
struct RowsQ6 {
    // (a wave keeps one block of a row: with two the kernel spilled, at 128 registers. Rows of 17 .. 32 blocks in two parts against
    // that, at one / four / eight tokens: 16384 x 8192 34.0 34.2 37.0 -> 29.1 28.9 31.1 us, 2 x 8192 x 6144 31.3 32.9 35.9 -> 26.9 27.5 29.8, 4096 x
    // 5120 12.6 13.1 16.5 -> 11.8 12.2 13.8, 2560 x 6912 11.2 12.2 15.5 -> 12.2 12.5 14.1)
    static constexpr uint32_t BLOCK = 224, CHUNKS = 14, SLOTS = 2, MOST = 1;
    static constexpr bool MINS = false, RAGGED = false, SPLIT = false;
    static const char *name() { return "matvec_q6_k"; }
    static __device__ __forceinline__ uint32_t chunk_at(uint32_t, uint32_t b, uint32_t c, uint32_t) { return BLOCK * b + 16u * c; }
    static __device__ __forceinline__ void multiply(const uint8_t *slot, uint32_t l16, uint32_t g, uint32_t, const f16x8 (&xf)[8], const f16x8 &, const float (&inv)[2], f32x4 &out) {
        const uint8_t *row = slot + BLOCK * l16;
        const u32x4 sc = *reinterpret_cast<const u32x4 *>(row + 192u);
        const float d = half_bits_to_float(*reinterpret_cast<const uint16_t *>(row + 208u));
        const uint32_t sel = g >= 2u ? 0x04030401u : 0x04020400u;  // the lane's half of a unit, of two units
        f32x4 sums[4] = {}, rest = {0.f, 0.f, 0.f, 0.f};  // of two units' rounded products each, and of what that left: shorter sums
#pragma unroll
        for (uint32_t n = 0; n < 2; n++) {
            const u32x2 l[2] = {*reinterpret_cast<const u32x2 *>(row + 64u * n + 8u * g), *reinterpret_cast<const u32x2 *>(row + 64u * n + 32u + 8u * g)};
            const u32x2 h = *reinterpret_cast<const u32x2 *>(row + 128u + 32u * n + 8u * g);
#pragma unroll
            for (uint32_t c = 0; c < 4; c++) {
                // Two units' scales: 1152 + value in the mantissa of 1024, less 1152.
                const f16x2 s2 = as_f16(__builtin_amdgcn_perm(0x64u, sc[2 * n + (c >> 1)] ^ 0x80808080u, sel)) + f16x2{(_Float16)-1152.f, (_Float16)-1152.f};
                const f16x2 s = {s2[c & 1], s2[c & 1]};
                const f16x2 minus = c < 2 ? f16x2{(_Float16)-1056.f, (_Float16)-1056.f} : f16x2{(_Float16)-96.f, (_Float16)-96.f};
                f16x2 high[4], low[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t w = l[c & 1][e >> 1], f = h[e >> 1];
                    const uint32_t nib = (e & 1) ? w >> 8 : w;
                    // Low nibbles under the exponent of 1024, high ones under that of 64; the two upper bits above them.
                    const int up = (c < 2 ? 4 : 8) - 2 * (int)c - 8 * (e & 1);
                    const uint32_t two = up >= 0 ? f << (up & 31) : f >> (-up & 31);
                    const uint32_t v = c < 2 ? and_or(nib, 0x000f000fu, 0x64006400u) | (two & 0x00300030u) : and_or(nib, 0x00f000f0u, 0x54005400u) | (two & 0x03000300u);
                    const f16x2 q = as_f16(v) + minus;
                    high[e] = q * s;
                    low[e] = fma2(q, s, -high[e]);
                }
                sums[2 * n + (c & 1)] = mfma(xf[4 * n + c], pack(high[0], high[1], high[2], high[3]), sums[2 * n + (c & 1)]);
                rest = mfma(xf[4 * n + c], pack(low[0], low[1], low[2], low[3]), rest);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) out[e] = fmaf(inv[e >> 1] * d, ((sums[0][e] + sums[1][e]) + (sums[2][e] + sums[3][e])) + rest[e], out[e]);
    }
};

// Q3_K (repacked into eight 16-byte units a block: two words of 2-bit values, the third bits, two
// scales - 32 and d): a weight is d * s * (q - 4), the product exact in f16. Blocks are 128 bytes, so their
// units are permuted by the row: unpermuted, sixteen rows' reads would meet in two banks.
struct RowsQ3 {
    static constexpr uint32_t BLOCK = 128, CHUNKS = 8, SLOTS = 3, MOST = 2;
    static constexpr bool MINS = false, RAGGED = false, SPLIT = false;
    static const char *name() { return "matvec_q3_k"; }
    static __device__ __forceinline__ uint32_t chunk_at(uint32_t, uint32_t b, uint32_t c, uint32_t row) { return BLOCK * b + 16u * (c ^ (row & 7u)); }
    static __device__ __forceinline__ void multiply(const uint8_t *slot, uint32_t l16, uint32_t g, uint32_t, const f16x8 (&xf)[8], const f16x8 &, const float (&inv)[2], f32x4 &out) {
        const uint8_t *row = slot + BLOCK * l16;
        const uint32_t sel = g >= 2u ? 0x04010401u : 0x04000400u, shift = 4u * (g & 1u);
        f32x4 sums[2] = {};
        float d = 0.f;
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(row + 16u * (u ^ (l16 & 7u)));
            if (u == 0) d = half_bits_to_float(v.w >> 16);
            const f16x2 s = as_f16(__builtin_amdgcn_perm(0x64u, v.w ^ 0x8080u, sel)) + f16x2{(_Float16)-1152.f, (_Float16)-1152.f};
            // Positions 8 g .. + 3: bits 0, 1 of the word's bytes; + 4 .. + 7: bits 2, 3, under the exponent of 256.
            const uint32_t t = (g >= 2u ? v.y : v.x) >> shift, z = v.z >> (2u * g), t8 = t >> 8;
            const f16x2 q0 = as_f16(and_or(t, 0x00030003u, 0x64006400u) | ((z << 2) & 0x00040004u)), q1 = as_f16(and_or(t8, 0x00030003u, 0x64006400u) | ((z >> 6) & 0x00040004u));
            const f16x2 q2 = as_f16(and_or(t, 0x000c000cu, 0x5c005c00u) | ((z << 3) & 0x00100010u)), q3 = as_f16(and_or(t8, 0x000c000cu, 0x5c005c00u) | ((z >> 5) & 0x00100010u));
            const f16x2 m0 = {(_Float16)-1028.f, (_Float16)-1028.f}, m2 = {(_Float16)-260.f, (_Float16)-260.f};
            sums[u & 1] = mfma(xf[u], pack((q0 + m0) * s, (q1 + m0) * s, (q2 + m2) * s, (q3 + m2) * s), sums[u & 1]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) out[e] = fmaf(inv[e >> 1] * d, sums[0][e] + sums[1][e], out[e]);
    }
};

// Q8_0 split rows (k signed bytes, then k / 32 f16 scales): in a slot a row's 256 bytes and its eight
// scales. The scale, eleven bits of its own, meets a unit's sums.
struct RowsQ8 {
    static constexpr uint32_t BLOCK = 272, CHUNKS = 17, SLOTS = 2, MOST = 2;
    static constexpr bool MINS = false, RAGGED = true, SPLIT = true;
    static const char *name() { return "matvec_q8_0"; }
    static __device__ __forceinline__ uint32_t chunk_at(uint32_t k, uint32_t b, uint32_t c, uint32_t) { return c < 16u ? 256u * b + 16u * c : k + 16u * b; }
    static __device__ __forceinline__ void multiply(const uint8_t *slot, uint32_t l16, uint32_t g, uint32_t units, const f16x8 (&xf)[8], const f16x8 &, const float (&inv)[2], f32x4 &out) {
        const uint8_t *row = slot + BLOCK * l16;
        const u32x4 sc = *reinterpret_cast<const u32x4 *>(row + 256u);
        f32x4 block[2] = {};
        const f16x2 minus = {(_Float16)-1152.f, (_Float16)-1152.f};
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            if (u >= units) break;
            u32x2 w = *reinterpret_cast<const u32x2 *>(row + 32u * u + 8u * g);
            w.x ^= 0x80808080u;
            w.y ^= 0x80808080u;
            const f32x4 r = mfma(xf[u], pack(as_f16(__builtin_amdgcn_perm(0x64u, w.x, 0x04020400u)) + minus, as_f16(__builtin_amdgcn_perm(0x64u, w.x, 0x04030401u)) + minus,
                as_f16(__builtin_amdgcn_perm(0x64u, w.y, 0x04020400u)) + minus, as_f16(__builtin_amdgcn_perm(0x64u, w.y, 0x04030401u)) + minus), f32x4{0.f, 0.f, 0.f, 0.f});
            const float d = half_bits_to_float((u & 1u) ? sc[u >> 1] >> 16 : sc[u >> 1] & 0xffffu);
#pragma unroll
            for (int e = 0; e < 4; e++) block[u & 1][e] = fmaf(d, r[e], block[u & 1][e]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) out[e] = fmaf(inv[e >> 1], block[0][e] + block[1][e], out[e]);
    }
};

// A wave's slots of weights: the first has a place of its own, the others lie in the operands' place, which is
// free once they are in registers.
template <class F> constexpr uint32_t shared_bytes() {
    constexpr uint32_t operands = F::MINS ? OPERANDS : SUMS_AT, slots = (F::SLOTS - 1u) * 16u * F::BLOCK;
    return operands > slots ? operands : slots;
}
template <class F> constexpr uint32_t wave_bytes() { return shared_bytes<F>() + 16u * F::BLOCK; }

// NB: the most blocks of 256 weights a wave takes of a row. LONG: q.parts workgroups share a tile, each over
// its share of the row's blocks, and leave their sums in q.partial.
template <class F, int NB, int TEAMS, bool ACT, bool LONG>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4))) void matvec_mfma_rows_kernel(const float *first_x, const uint8_t *first_w, const float *first_norm_w,
    uint32_t k_flags, uint32_t xr, uint32_t row_bytes, uint32_t rows, uint32_t half_at, uint32_t groups_left, uint32_t whole_rounds, uint32_t counts, RowsArgs q) {
    // (ahead of the struct, in registers when the wave starts: what the first loads of inputs and weights are addressed by; see
    // MV_FIRST. Some share a word: launch_nb. With the other matrix-core kernels' and the sums', four tokens through eight layers of
    // 4096 x 14336 Q4_K, 597 -> 582 us a step.)
    q.a.x = first_x, q.a.w = first_w, q.a.norm_w = first_norm_w, q.a.k = k_flags & 0xffffffu, q.a.flags = k_flags >> 24, q.a.xr = xr, q.a.row_bytes = row_bytes;
    q.a.rows = rows, q.a.half = half_at, q.groups = groups_left & 0xffffu, q.left = groups_left >> 16, q.rounds = whole_rounds;
    q.a.m = counts & 15u, q.split = counts >> 4 & 1u, q.parts = counts >> 8 & 255u, q.blocks = counts >> 16;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float lds_part[2][WAVES][128];  // [round parity][wave][2 lane + token of the lane's two]
    __shared__ float lds_ss[WAVES][8];
    __shared__ float lds_before[4][128];       // [output tile of the round]: what the outputs hold, for a step that accumulates
    static_assert(!LONG || (NB == 1 && TEAMS == 1), "a part is a block a wave");
    constexpr uint32_t SLOT = 16u * F::BLOCK, PIECES = 16u * F::CHUNKS;
    constexpr int LOADS = (int)((PIECES + 63u) / 64u);
    constexpr uint32_t SLOTS = F::SLOTS, WAVE_BYTES = wave_bytes<F>();
    const MvArgs &a = q.a;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool pair = (a.flags & FLAG_SILU_PAIR) != 0, norm = (a.flags & FLAG_NORM) != 0, accumulate = !LONG && (a.flags & FLAG_ACCUMULATE) != 0;

    // Short rows leave a tile to a half, a quarter, ... of the waves: a team. The wave's blocks of every
    // row of its team's tiles.
    constexpr uint32_t teams = TEAMS, members = WAVES / TEAMS;
    const uint32_t team = wave / members, member = wave % members;
    const uint32_t walker = LONG ? blockIdx.x / q.parts : blockIdx.x, kpart = LONG ? blockIdx.x % q.parts : 0u;
    const uint32_t start = LONG ? kpart * q.blocks / q.parts : 0u, blocks = LONG ? (kpart + 1u) * q.blocks / q.parts - start : q.blocks;
    const uint32_t first = start + member * blocks / members, mine = start + (member + 1u) * blocks / members - first;
    // ---- the wave's blocks of the tokens' inputs, four positions a lane and token, asked for before anything else.
    // With several teams the first two share the tokens out between them and all read what they leave.
    // (Tokens in groups of two or four without branches between them, so that their chains overlap; an
    // absent one reads zeros.)
    constexpr bool shared = teams > 1u;
    const uint32_t half = a.m > 4u ? 4u : 2u, base = shared ? team * half : 0u;  // first token the wave stages
    const uint32_t staged = !shared ? a.m : team < 2u && base < a.m ? half : 0u;
    f32x4 xv[NB][8], gv[NB];
    // (one buffer from the first token to the end of the last: a token past it reads zeros; positions past the
    // end of a ragged row are asked for past it)
    const __amdgpu_buffer_rsrc_t xbuf = make_buffer(a.x + (size_t)base * a.xr, base < a.m ? ((a.m - 1u - base) * a.xr + a.k) * 4u : 0u);
    uint32_t at[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        at[b] = 1024u * (first + b) + 16u * lane;
        if (F::RAGGED) at[b] = at[b] < 4u * a.k ? at[b] : kNowhere;
    }
    auto load_tokens = [&](auto from, auto to) __attribute__((always_inline)) {
#pragma unroll
        for (int t = from; t < to; t++)
#pragma unroll
            for (int b = 0; b < NB; b++) xv[b][t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, F::RAGGED ? (at[b] + 4u * a.xr * t) | (at[b] & kNowhere) : at[b] + 4u * a.xr * t, 0, 0));
    };
    constexpr std::integral_constant<int, 0> T0{};
    constexpr std::integral_constant<int, 2> T2{};
    constexpr std::integral_constant<int, 4> T4{};
    constexpr std::integral_constant<int, 8> T8{};
    if (staged > 0u) load_tokens(T0, T2);
    if (staged > 2u) load_tokens(T2, T4);
    if (staged > 4u) load_tokens(T4, T8);
    if (norm) {
#pragma unroll
        for (int b = 0; b < NB; b++) gv[b] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(make_buffer(a.norm_w, a.k * 4u), at[b], 0, 0));
    }

    // The workgroup's weight tiles: output tiles b, b + G, ...; with SILU_PAIR the gate tile
    // and then the up tile of each. When the output tiles left over after whole rounds are at most half
    // as many as the workgroups, two workgroups share each, eight rows apiece.
    const uint32_t per = pair ? 2u : 1u;
    const bool extra = walker < (q.split ? 2u * q.left : q.left);
    const uint32_t count = per * (q.rounds + (extra ? 1u : 0u));
    const uint32_t last_out = 16u * (q.rounds * q.groups + (q.split ? walker >> 1 : walker)) + (q.split ? 8u * (walker & 1u) : 0u);
    auto output = [&](uint32_t p) { return pair ? p >> 1 : p; };
    auto out0 = [&](uint32_t p) { return output(p) < q.rounds ? 16u * (walker + output(p) * q.groups) : last_out; };
    auto rows_of = [&](uint32_t p) {
        const uint32_t at = out0(p), left = at < a.rows ? a.rows - at : 0u, most = (q.split && output(p) >= q.rounds) ? 8u : 16u;
        return left < most ? left : most;
    };

    // ---- weights: a block of the tile's sixteen rows at a time, 16-byte pieces in the order of the
    // rows into one of the wave's slots. Pieces of rows the tile does not have are past the buffer's end.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
    const uint32_t operands_at = wave * WAVE_BYTES;
    auto slot_at = [&](uint32_t s) { return operands_at + (s == 0u ? shared_bytes<F>() : (s - 1u) * SLOT); };
    uint32_t piece_at[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
        const uint32_t i = 64u * j + lane;
        piece_at[j] = i / F::CHUNKS * a.row_bytes + F::chunk_at(a.k, first, i % F::CHUNKS, i / F::CHUNKS);
    }
    uint32_t fetch_tile = team, fetch_block = 0, fetch_slot = 0;
    __amdgpu_buffer_rsrc_t wbuf;
    auto next_tile = [&]() __attribute__((always_inline)) {
        const bool real = fetch_tile < count && mine > 0u;
        const uint32_t row = __builtin_amdgcn_readfirstlane(real ? out0(fetch_tile) + ((pair && (fetch_tile & 1u)) ? a.half : 0u) : 0u);
        wbuf = make_buffer(a.w + (size_t)row * a.row_bytes, __builtin_amdgcn_readfirstlane(real ? rows_of(fetch_tile) * a.row_bytes : 0u));
    };
    next_tile();
    auto fetch = [&]() __attribute__((always_inline)) {
        const uint32_t dst = lds0 + slot_at(fetch_slot), block_at = (F::SPLIT ? 256u : F::BLOCK) * fetch_block;
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            // (of split rows the scales of the next block are 16 bytes on, not 256)
            const uint32_t at = F::SPLIT && (64u * j + lane) % F::CHUNKS == 16u ? piece_at[j] - 240u * fetch_block : piece_at[j];
            if (64u * (j + 1u) <= PIECES || lane < PIECES - 64u * j) load_lds_b128(wbuf, dst + 1024u * j, at, block_at);
        }
        fetch_slot = fetch_slot + 1u == SLOTS ? 0u : fetch_slot + 1u;
        if (++fetch_block >= mine) {
            fetch_block = 0;
            fetch_tile += teams;
            next_tile();
        }
    };

    // ---- the tokens' operands
    fetch();
    // The norm's factor is a token's own and is left to the outputs, unless it goes through the
    // activation.
    auto square_sums = [&](auto from, auto to) __attribute__((always_inline)) {
        constexpr int G = to - from;
        float ss[G];
#pragma unroll
        for (int t = 0; t < G; t++) {
            ss[t] = 0.f;
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) ss[t] = fmaf((uint32_t)b < mine ? xv[b][from + t][e] : 0.f, xv[b][from + t][e], ss[t]);
        }
        const float sum = over_tokens<G>(ss, lane, [](float x, float y) { return x + y; });
        if (lane < (uint32_t)G) lds_ss[wave][base + from + lane] = sum;
    };
    if (norm) {
        if (shared && lane < 8u) lds_ss[wave][lane] = 0.f;
        if (staged > 2u) square_sums(T0, T4);
        else if (staged > 0u) square_sums(T0, T2);
        if (staged > 4u) square_sums(T4, T8);
    }
    // One over the root mean square of token t, behind a barrier after the above.
    auto norm_scale = [&](uint32_t t) {
        float total = lds_ss[0][t];
#pragma unroll
        for (uint32_t w = 1; w < WAVES; w++) total += lds_ss[w][t];
        return 1.0f / sqrtf(total / (float)a.k + a.eps);
    };
    const bool early = ACT && norm;
    if constexpr (ACT) {
        if (early && !LONG) lds_barrier();
#pragma unroll
        for (int t = 0; t < 8; t++) {
            if ((uint32_t)t >= staged) break;
            const float scale = !early ? 1.0f : LONG ? q.partial[kScales + base + t] : norm_scale(base + t);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                if (norm) xv[b][t] *= gv[b];
#pragma unroll
                for (int e = 0; e < 4; e++) xv[b][t][e] = silu_f(xv[b][t][e] * scale / a.act_div);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) gv[b] = f32x4{1.f, 1.f, 1.f, 1.f};
    }
    f16x8 xf[NB][8], xsum[NB];
    float inv[NB][2];
    uint8_t *const place = lds + operands_at + (lane >> 1) * GROUP + 8u * (lane & 1u);
    auto stage = [&](int b, auto from, auto to) __attribute__((always_inline)) {
        constexpr int G = to - from;
        f32x4 v[G];
        float big[G];
#pragma unroll
        for (int t = 0; t < G; t++) {
            v[t] = xv[b][from + t];
            if (norm) v[t] *= gv[b];
            big[t] = fmaxf(fmaxf(fabsf(v[t][0]), fabsf(v[t][1])), fmaxf(fabsf(v[t][2]), fabsf(v[t][3])));
        }
        // The power of two that puts the block's largest magnitude of a token in [2^14, 2^15) (2^126 at most).
        const uint32_t exponent = __float_as_uint(over_tokens<G>(big, lane, [](float x, float y) { return fmaxf(x, y); })) >> 23;
        uint32_t up = 268u - exponent;
        up = (up > 253u ? 253u : up) << 23;
        if (lane < (uint32_t)G) *reinterpret_cast<float *>(lds + operands_at + INVERSE_AT + 4u * lane) = __uint_as_float((254u << 23) - up);
        // (An infinity's rounding leaves inf - inf: INFINITE makes that a zero. The finite inputs of its block, under the scale
        // that the infinity's exponent gives, vanish beside it. One branch a group of tokens, so that their chains still overlap.)
        auto put = [&](auto infinite) __attribute__((always_inline)) {
            constexpr bool INFINITE = decltype(infinite)::value;
            auto rest = [](float v, float scale, _Float16 rounded) { return INFINITE && !(fabsf((float)rounded) <= 65504.f) ? (_Float16)0.f : (_Float16)fmaf(v, scale, -(float)rounded); };
#pragma unroll
            for (int t = 0; t < G; t++) {
                const uint32_t bits = __builtin_amdgcn_readlane(up, t);
                const float scale = __uint_as_float(bits);
                _Float16 hi[4], lo[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    hi[e] = (_Float16)(v[t][e] * scale);
                    lo[e] = rest(v[t][e], scale, hi[e]);
                }
                *reinterpret_cast<f16x4 *>(place + 32u * t) = f16x4{hi[0], hi[2], hi[1], hi[3]};
                *reinterpret_cast<f16x4 *>(place + 32u * t + 16u) = f16x4{lo[0], lo[2], lo[1], lo[3]};
                if (F::MINS) {
                    // The unit's sum, over 32, the same way: half lane / 8 of the sums' rows.
                    float sum = (v[t][0] + v[t][1]) + (v[t][2] + v[t][3]);
                    sum = add_dpp<0xB1>(sum);
                    sum = add_dpp<0x4E>(sum);
                    sum = add_dpp<0x141>(sum);
                    const float part = scale * 0.03125f;
                    const _Float16 sum_hi = (_Float16)(sum * part), sum_lo = rest(sum, part, sum_hi);
                    if ((lane & 7u) == 0u) {
                        *reinterpret_cast<_Float16 *>(lds + operands_at + SUMS_AT + 32u * t + 2u * (lane >> 3)) = sum_hi;
                        *reinterpret_cast<_Float16 *>(lds + operands_at + SUMS_AT + 32u * t + 16u + 2u * (lane >> 3)) = sum_lo;
                    }
                }
            }
        };
        put(std::false_type{});
        if (__ballot(exponent == 255u)) put(std::true_type{});
    };
    // Operand row l16 is token l16 / 2's, from where the token lies (an absent token's rows are whatever lies
    // there: they meet no other token's); positions of the sums' rows past the eight units are zeros. The lane's
    // results are tokens 2 g and 2 g + 1.
    auto read = [&](int b, uint32_t from, uint32_t row, uint32_t inverse_from, uint32_t token, bool keep) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            const f16x8 got = *reinterpret_cast<const f16x8 *>(lds + from + (4u * u + g) * GROUP + 16u * row);
            xf[b][u] = keep ? xf[b][u] : got;
        }
        if (F::MINS) {
            u32x4 sums = *reinterpret_cast<const u32x4 *>(lds + from + SUMS_AT + 16u * row);
#pragma unroll
            for (int e = 0; e < 4; e++) sums[e] = g == 0u ? sums[e] : 0u;
            xsum[b] = keep ? xsum[b] : __builtin_bit_cast(f16x8, sums);
        }
        const float2 two = *reinterpret_cast<const float2 *>(lds + inverse_from + INVERSE_AT + 4u * token);
        inv[b][0] = two.x;
        inv[b][1] = two.y;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    if (shared) {
        if (staged > 2u) stage(0, T0, T4);
        else if (staged > 0u) stage(0, T0, T2);
        lds_barrier();
        const uint32_t from = l16 >= 2u * half ? 1u : 0u, inverse_from = 2u * g >= half ? 1u : 0u;
        read(0, (member + from * members) * WAVE_BYTES, (l16 - 2u * half * from) & 7u, (member + inverse_from * members) * WAVE_BYTES, (2u * g - half * inverse_from) & 3u, false);
        lds_barrier();  // the operands' place may be filled with weights
    } else {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if ((uint32_t)b >= mine) break;
            if (a.m <= 2u) stage(b, T0, T2);
            else stage(b, T0, T4);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            read(b, operands_at, l16 & 7u, operands_at, (2u * g) & 3u, false);
            if (a.m > 4u) {
                const float low[2] = {inv[b][0], inv[b][1]};
                stage(b, T4, T8);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                read(b, operands_at, l16 & 7u, operands_at, (2u * g) & 3u, l16 < 8u);
                inv[b][0] = g < 2u ? low[0] : inv[b][0];
                inv[b][1] = g < 2u ? low[1] : inv[b][1];
            }
        }
    }
#pragma unroll
    for (uint32_t i = 1; i + 1u < SLOTS; i++) fetch();

    float held = 0.f;  // the gate tile's result, until the up tile's arrives
    const uint32_t my_row = tid & 15u, my_token = (tid >> 4) & 7u;
    // The members' partial sums of the tile of a team, of the thread's row and token.
    auto team_sum = [&](const float *part, uint32_t of) __attribute__((always_inline)) {
        const float *src = part + of * members * 128u + 2u * ((my_token >> 1) * 16u + my_row) + (my_token & 1u);
        float v[members];
#pragma unroll
        for (uint32_t w = 0; w < members; w++) v[w] = src[w * 128u];
#pragma unroll
        for (uint32_t step = 1; step < members; step *= 2u)
#pragma unroll
            for (uint32_t w = 0; w + step < members; w += 2u * step) v[w] += v[w + step];
        const float sum = v[0];
        return norm && !early && !LONG ? sum * norm_scale(my_token) : sum;
    };
    // Adds up a round's tiles, behind the barrier that follows their multiply: an output tile is two
    // waves' to add, others from one output tile to the next. (Four teams' four output tiles a round use
    // every place of lds_before: they stay with the same waves, or those of the next round would fill a place that is still read.)
    constexpr uint32_t adders = teams == 4u ? 3u : 7u;
    auto sum_up = [&](uint32_t round) __attribute__((always_inline)) {
        const float *part = &lds_part[round & 1u][0][0];
        const bool whole = pair && teams > 1u;  // the round has both tiles of an output
        for (uint32_t of = 0; of < teams; of += whole ? 2u : 1u) {
            const uint32_t p = round * teams + of, o = output(p);
            if (p >= count || (wave >> 1) != (o & adders)) continue;
            const float sum = team_sum(part, of);
            if (LONG) {
                if (my_token < a.m && my_row < rows_of(p)) store_apart(q.partial + kSums + ((size_t)((pair ? 2u : 1u) * kpart + (pair ? p & 1u : 0u)) * 8u + my_token) * a.rows + out0(p) + my_row, sum);
                if (norm && !early && round == 0u && walker == 0u && p == 0u && my_row == 0u) {
                    float total = lds_ss[0][my_token];
#pragma unroll
                    for (uint32_t w = 1; w < WAVES; w++) total += lds_ss[w][my_token];
                    store_apart(q.partial + 8u * kpart + my_token, total);
                }
                continue;
            }
            if (pair && !whole && !(p & 1u)) {
                held = sum;
                continue;
            }
            float v = whole ? silu_f(sum) * team_sum(part, of + 1u) : pair ? silu_f(held) * sum : sum;
            if (accumulate) {
                if (mine > 0u) wait_loads<LOADS>();  // (one block's loads have been issued behind it)
                else wait_loads<0>();
                v += lds_before[o & 3u][tid & 127u];
            }
            if (my_token < a.m && my_row < rows_of(p)) store_apart(a.out + (size_t)my_token * a.out_stride + a.col0 + out0(p) + my_row, v);
        }
    };
    uint32_t slot = 0;
    const uint32_t rounds = (count + teams - 1u) / teams;
    for (uint32_t round = 0; round < rounds; round++) {
        if (accumulate) {
            for (uint32_t of = 0; of < teams; of++) {
                const uint32_t p = round * teams + of, o = output(p);
                if (p >= count || (wave >> 1) != (o & adders) || (pair && (p & 1u))) continue;
                const bool there = my_token < a.m && my_row < rows_of(p);
                const uint32_t at = there ? (my_token * a.out_stride + a.col0 + out0(p) + my_row) * 4u : kNowhere;
                load_lds_b32(make_buffer(a.out, kOutBytes), (uint32_t)(uintptr_t)(lds_ptr)&lds_before[o & 3u][64u * (wave & 1u)], at);
            }
        }
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if ((uint32_t)b >= mine) break;
            fetch();
            wait_loads<(SLOTS - 1) * LOADS>();
            const uint32_t left = a.k / 32u - 8u * (first + b), units = !F::RAGGED || left >= 8u ? 8u : left;
            F::multiply(lds + slot_at(slot), l16, g, units, xf[b], xsum[b], inv[b], acc);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            slot = slot + 1u == SLOTS ? 0u : slot + 1u;
        }
        // (a token's two rows: its rounded inputs and what the rounding left)
        *reinterpret_cast<float2 *>(&lds_part[round & 1u][wave][2u * lane]) = float2{acc[0] + acc[1], acc[2] + acc[3]};
        lds_barrier();
        sum_up(round);
    }
    wait_loads<0>();  // nothing may still land in LDS once the workgroup is gone
}

// The outputs of a step over rows in parts: the parts' sums in the order of their blocks, the norm's
// factor, the SILU_PAIR / ACCUMULATE epilogue. One thread an output.
template <bool PAIR>
__global__ __launch_bounds__(256) void matvec_mfma_rows_sum_kernel(const float *partial, float *out, uint32_t rows, uint32_t m, uint32_t out_stride, uint32_t accumulate, uint32_t parts, uint32_t norm, uint32_t k, float eps) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, row = i % rows, t = i / rows;
    if (t >= m) return;
    constexpr uint32_t per = PAIR ? 2u : 1u;
    const float *src = partial + kSums + (size_t)t * rows + row;
    const size_t plane = (size_t)8u * rows;
    float *o = out + (size_t)t * out_stride + row;
    // Every load first: the parts were written by other workgroups and come from memory.
    float first[kMaxParts], second[kMaxParts], squares[kMaxParts];
#pragma unroll
    for (uint32_t p = 0; p < kMaxParts; p++) {
        first[p] = p < parts ? src[per * p * plane] : 0.f;
        second[p] = (PAIR && p < parts) ? src[(per * p + 1u) * plane] : 0.f;
        squares[p] = (norm && p < parts) ? partial[8u * p + t] : 0.f;
    }
    const float before = accumulate ? *o : 0.f;
    float sum = first[0], up = second[0], ss = squares[0];
#pragma unroll
    for (uint32_t p = 1; p < kMaxParts; p++) {
        sum += first[p];
        up += second[p];
        ss += squares[p];
    }
    if (norm) {
        const float scale = 1.0f / sqrtf(ss / (float)k + eps);
        sum *= scale;
        up *= scale;
    }
    const float v = PAIR ? silu_f(sum) * up : sum;
    *o = accumulate ? before + v : v;
}

template <class F, int NB, int TEAMS, bool ACT, bool LONG>
zhip_result launch_nb(const Dispatch &d, const RowsArgs &q) {
    constexpr int bytes = (int)(WAVES * wave_bytes<F>());
    if (!lds_opt_in<matvec_mfma_rows_kernel<F, NB, TEAMS, ACT, LONG>, bytes>()) return fail(d, ZHIP_E_GPU, "%s: cannot reserve %d bytes of LDS", F::name(), bytes);
    if (!MV_HOLDS(q.a) || q.a.m > 15u || q.parts > 255u || (q.blocks | q.groups | q.left) > 0xffffu)
        return fail(d, ZHIP_E_GPU, "%s: %u tokens, %u blocks in %u parts, %u workgroups, %u tiles left", F::name(), q.a.m, q.blocks, q.parts, q.groups, q.left);
    hipLaunchKernelGGL((matvec_mfma_rows_kernel<F, NB, TEAMS, ACT, LONG>), dim3(q.groups * q.parts), dim3(THREADS), bytes, d.stream, q.a.x, q.a.w, q.a.norm_w, q.a.k | q.a.flags << 24, q.a.xr,
        q.a.row_bytes, q.a.rows, q.a.half, q.groups | q.left << 16, q.rounds, q.a.m | q.split << 4 | q.parts << 8 | q.blocks << 16, q);
    return check_launch(d, F::name());
}

template <class F, int NB, int TEAMS, bool LONG>
zhip_result launch_act(const Dispatch &d, const RowsArgs &q) {
    return q.a.act_div > 0.f ? launch_nb<F, NB, TEAMS, true, LONG>(d, q) : launch_nb<F, NB, TEAMS, false, LONG>(d, q);
}

template <class F>
zhip_result launch_format(const Dispatch &d, const MvArgs &a) {
    const bool pair = (a.flags & FLAG_SILU_PAIR) != 0, norm = (a.flags & FLAG_NORM) != 0;
    const uint32_t blocks = (a.k + 255u) / 256u, tiles = (a.rows + 15u) / 16u;
    const uint32_t parts = blocks > F::MOST * WAVES ? (blocks + WAVES - 1u) / WAVES : 1u;
    const uint32_t most = std::min((uint32_t)d.dev->compute_units, 0xffffu) / parts;  // (the count has half a word of the kernel's parameters)
    if (most == 0u) return fail(d, ZHIP_E_GPU, "%s: %d compute units for %u parts of a row", F::name(), d.dev->compute_units, parts);
    const uint32_t groups = tiles < most ? (2u * tiles <= most ? 2u * tiles : tiles) : most;
    const bool halves = tiles < groups;  // every workgroup takes eight outputs of one tile
    const uint32_t left = halves ? tiles : tiles % groups, count = (halves ? 1u : (tiles + groups - 1u) / groups) * (pair ? 2u : 1u);
    RowsArgs q{a, blocks, groups, halves ? 0u : tiles / groups, left, (halves || 2u * left <= groups) ? 1u : 0u, parts, nullptr};
    if (parts > 1u) {
        const uint64_t bytes = (kSums + (uint64_t)parts * (pair ? 2u : 1u) * 8u * a.rows) * sizeof(float);
        if (!d.work) return fail(d, ZHIP_E_GPU, "%s: no workspace", F::name());
        if (zhip_result r = d.work->reserve(d, bytes)) return r;
        q.partial = reinterpret_cast<float *>(d.work->data);
        if (norm && a.act_div > 0.f) {
            if (zhip_result r = launch_matvec_parts_scales(d, F::name(), a, q.partial + kScales)) return r;
        }
        if (zhip_result r = launch_act<F, 1, 1, true>(d, q)) return r;
        const dim3 sums((a.rows * a.m + 255u) / 256u);
        if (pair) hipLaunchKernelGGL(matvec_mfma_rows_sum_kernel<true>, sums, dim3(256), 0, d.stream, q.partial, a.out + a.col0, a.rows, a.m, a.out_stride, a.flags & FLAG_ACCUMULATE, parts, norm && a.act_div <= 0.f, a.k, a.eps);
        else hipLaunchKernelGGL(matvec_mfma_rows_sum_kernel<false>, sums, dim3(256), 0, d.stream, q.partial, a.out + a.col0, a.rows, a.m, a.out_stride, a.flags & FLAG_ACCUMULATE, parts, norm && a.act_div <= 0.f, a.k, a.eps);
        return check_launch(d, F::name());
    }
    if constexpr (F::MOST > 1u) {
        if (blocks > WAVES) return launch_act<F, 2, 1, false>(d, q);
    }
    if (blocks > WAVES / 2u) return launch_act<F, 1, 1, false>(d, q);
    if (blocks > WAVES / 4u || count < 4u) return launch_act<F, 1, 2, false>(d, q);
    return launch_act<F, 1, 4, false>(d, q);
}

}  // namespace

// Whether the kernel can run the (already validated) arguments: rows of up to eight parts, and inputs and (where it adds
// to them) outputs that its 32-bit offsets reach, of eight tokens so that the route is the same at every width.
bool matvec_mfma_rows_accepts(const MvArgs &a) {
    const uint64_t x_end = (7ull * a.xr + a.k) * 4u, out_end = (7ull * a.out_stride + a.col0 + a.rows) * 4u;
    return a.m >= 1u && a.m <= 8u && a.k <= kMaxParts * WAVES * 256u && x_end < kNowhere && (!(a.flags & FLAG_ACCUMULATE) || out_end <= kOutBytes);
}
zhip_result launch_matvec_mfma_rows(const Dispatch &d, const MvArgs &a, int type) {
    switch (type) {
    case 3: return launch_format<RowsQ3>(d, a);
    case 4: return launch_format<RowsQ45<false>>(d, a);
    case 5: return launch_format<RowsQ45<true>>(d, a);
    case 6: return launch_format<RowsQ6>(d, a);
    default: return launch_format<RowsQ8>(d, a);
    }
}

}  // namespace zhip
