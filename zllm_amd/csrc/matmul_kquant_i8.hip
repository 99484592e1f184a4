// matmul_q3_k / matmul_q4_k / matmul_q5_k / matmul_q6_k over whole, unsliced k: a planner's prefill
// step on activations rounded to 8-bit blocks (quantize_q8), as src/kernels/matmul_quant.wgsl
// defines it:
//   out[t][col0 + j] = sum over 256-weight blocks of dx * (d * sum(s * q * qx) - dmin * sum(m * qx))
// with d, dmin and dx f32 and everything under the sums integer and exact.
//
// What bounds it: vector issue. A matrix instruction of 32 x 32 x 32 takes a SIMD 15 - 20 ns (the
// clock falls with what the operands toggle) and up to five vector instructions hide behind it
// (two waves a SIMD: the instruction alone 16.0 ns, with four multiply-adds 14.4 - 16, with eight 20,
// with sixteen 35), but applying a unit's 6- or 8-bit scale to its sums, as this kernel's
// predecessor did, is sixteen multiply-adds a unit and tile. Here the scale goes into the weights,
// once for all the tokens of a tile: s * q as two signed bytes (Q3_K: one), each plane a matrix
// instruction, and the block's sum is (high << SHIFT) + low. The integers are exact either way.
//   Q4_K: s = 8 a + b with a, b < 8, so the planes are a * q and b * q, at most 105: one packed
//         16-bit multiply makes four bytes of a plane (no product carries into its neighbour).
//   Q5_K, Q6_K: the 16-bit product s * q (Q6_K: s * (q - 32)) cut into its bytes, the low one
//         signed (the high one rounded up to match).
//   Q3_K: s * (q - 4) lies in -124 .. 128 and its negative in a byte: a lookup of the eight
//         possible products by byte permute, one plane, d negated.
// Q4_K and Q5_K minimums: one f16 instruction a tile and block, the tokens' sums over half units
// (exact, below 2048) against the minimums. With one token tile a wave (NT = 1) the converted
// weights would serve a single tile, and those two formats scale the sums after all.
//
// k is summed in four parts, blocks p * B / 4 .. of part p of B, each in its order, and the parts are
// added as ((p0 + p1) + p2) + p3, whatever the matrix and the step: neither how a prompt is cut into
// steps nor how a matrix is cut into launches changes an output's bits (but for the sign of a sum that is too small for a
// float: a wave with fewer steps than its workgroup adds zeros to it). A workgroup is S * RW waves.
// Wave w walks part w % S of k (S = 4), two of them (S = 2) or all four, closing each part's sums (S = 1), for rows 32 (w / S) .. + 31
// and the tile's 32 NT tokens, one 32-token tile of a block after the other with the block's
// converted weights in registers (64 VGPRs). Every part has a ring of three token tiles in LDS, filled
// two tiles ahead by whole-line direct loads that the part's RW waves share, and a wave's rows'
// blocks arrive in a slot of its own a block ahead. One barrier a tile where RW > 1, which leaves the
// loads in flight; the f32 end of a tile and block (five vector operations an output) is worked off
// between the next tile's matrix instructions.
//
// With few tokens over a tall matrix there is one workgroup of four walking waves a CU, one a SIMD, and nobody issues while it
// waits for an instruction's result; halving k gives every SIMD a second wave and leaves a wave's conversion its two token tiles: Q4_K 64 x
// 28672 x 4096 29.6 -> 24.7 us, Q6_K 64 x 24576 x 3072 30.6 -> 25.1, 256 x 19456 x 2560 56.0 -> 47.6, Q3_K 32 x 28672 x 4096 20.1 -> 16.4.
//
// Measured (us, weights from HBM, against the predecessor): Q4_K 512 x 4096 x 4096 37.9 -> 28.2, 512 x 28672 x
// 4096 232 -> 173, 512 x 4096 x 14336 115 -> 91, 128 x 4096 x 4096 17.3 -> 11.6, 64 x 4096 x 4096 9.7 -> 8.9;
// Q5_K 41.9 -> 32.9 / 259 -> 211 / 128 -> 101; Q6_K 53.7 -> 29.7 / 328 -> 187 / 171 -> 88; Q3_K
// 54.1 -> 19.2 / 302 -> 112 / 165 -> 60.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "decode.h"
#include "matmul_kquant_launch.h"

namespace zhip {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void *lds_ptr;

struct KqArgs {
    const uint8_t *qx;  // rows x k int8
    const uint8_t *w;   // rows of blocks as the loader lays them out
    const uint8_t *dx;  // rows x k / 256 f32
    float *out;
    uint32_t rows, n, k, col0, out_stride, accumulate, row_bytes;
    uint32_t qx_bytes, w_bytes, dx_bytes;
    uint32_t by_die;  // workgroups renumbered die by die
};

// A part's LDS: a ring of three token tiles, the tiles' scales, which are used a step later, and
// (where a format has minimums) the operands of two tiles' minimum instruction. A tile is eight runs
// of 1056 bytes: run i the 256 bytes of tokens i, i + 8, i + 16 and i + 24, with the neighbouring
// 16-byte chunks of the second and fourth exchanged, so that sixteen tokens' reads of the same
// chunk fall in sixteen bank groups at one immediate offset a unit.
constexpr uint32_t RING = 3, RUN = 1056, TILE_BYTES = 8 * RUN;
constexpr uint32_t DX_RING = 4, DX_BYTES = 256, DX_AT = RING * TILE_BYTES;
constexpr uint32_t SUMS_AT = DX_AT + DX_RING * DX_BYTES;
template <class P> constexpr uint32_t part_bytes() { return SUMS_AT + (P::HAS_MIN ? 2u * 1024u : 0u); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buffer(const uint8_t *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, (int)bytes, 0x00020000);
}
// One wave-wide load straight into LDS: lane l's bytes land at dst + 16 l (4 l). The destination
// reaches the load as a bare address, or the compiler would wait for every load in flight before
// each LDS read; the waits are this file's own.
__device__ __forceinline__ void load_lds_b128(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t offset, uint32_t uniform_offset) {
    uint32_t address = __builtin_amdgcn_readfirstlane(dst);
    asm volatile("" : "+s"(address));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)address, 16, offset, uniform_offset, 0, 0);
}
__device__ __forceinline__ void load_lds_b32(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t offset, uint32_t uniform_offset) {
    uint32_t address = __builtin_amdgcn_readfirstlane(dst);
    asm volatile("" : "+s"(address));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)address, 4, offset, uniform_offset, 0, 0);
}
// All but this wave's last LEFT loads have landed and its LDS reads have returned; then, where
// waves share what they loaded, the barrier.
template <int LEFT, bool SHARED>
__device__ __forceinline__ void step_end() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
    if (SHARED) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c));
}
// Four 16-bit values (of the even bytes' and the odd bytes' positions) plus 128, as two planes of
// signed bytes: value = 256 * high + low.
__device__ __forceinline__ uint32_t high_bytes(uint32_t even, uint32_t odd) { return __builtin_amdgcn_perm(odd, even, 0x07030501u); }
__device__ __forceinline__ uint32_t low_bytes(uint32_t even, uint32_t odd) { return __builtin_amdgcn_perm(odd, even, 0x06020400u) ^ 0x80808080u; }

// A format: BLOCK bytes; Raw, the bytes lane (row, h) reads of a block, positions 16 h .. + 15 of
// each of the eight 32-weight units; Scales, what is unpacked once a block; unit(): unit u's planes.
struct KqQ4 {
    static constexpr int TYPE = 4;
    static constexpr uint32_t BLOCK = 144;
    static constexpr int PLANES = 2, SHIFT = 3;
    static constexpr bool PERMUTED = false;
    static constexpr bool HAS_MIN = true;
    struct Raw {
        u32x4 h;     // d, dmin and the twelve scale bytes
        u32x4 q[4];  // 16 bytes of each 64-weight chunk: low nibbles unit 2 c, high 2 c + 1
    };
    struct Scales { uint32_t s[2]; };
    typedef f16x8 Mins;  // the eight minimums, the same for both halves of a unit
    static __device__ __forceinline__ void load(const uint8_t *blk, uint32_t, uint32_t h, uint32_t half, Raw &r) {
        if (half == 0u) r.h = *reinterpret_cast<const u32x4 *>(blk);
#pragma unroll
        for (uint32_t c = 2u * half; c < 2u * half + 2u; c++) r.q[c] = *reinterpret_cast<const u32x4 *>(blk + 16u + 32u * c + 16u * h);
    }
    // The eight 6-bit scales as bytes, and the minimums as f16 (src/ref/tensor.zig:94-98).
    static __device__ __forceinline__ Scales scales(const u32x4 &h) {
        Scales s;
        s.s[0] = h.y & 0x3f3f3f3fu;
        s.s[1] = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
        return s;
    }
    static __device__ __forceinline__ void header(const u32x4 &h, float &d, float &dmin, Mins &mins) {
        d = half_bits_to_float(h.x & 0xffffu);
        dmin = half_bits_to_float(h.x >> 16);
        const uint32_t m[2] = {h.z & 0x3f3f3f3fu, ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u)};
#pragma unroll
        for (int u = 0; u < 8; u++) mins[u] = (_Float16)(uint16_t)((m[u >> 2] >> (8 * (u & 3))) & 0xffu);
    }
    static __device__ __forceinline__ void factors(const Raw &r, float &d, float &dmin, Mins &mins) { header(r.h, d, dmin, mins); }
    static __device__ __forceinline__ Scales prepare(const Raw &r) { return scales(r.h); }
    // Unit u's weights as they are, and its scale.
    static __device__ __forceinline__ u32x4 plain(const Raw &r, uint32_t u) { return ((u & 1u) ? r.q[u >> 1] >> 4 : r.q[u >> 1]) & 0x0f0f0f0fu; }
    static __device__ __forceinline__ int scale(const Scales &sc, uint32_t u) { return (int)(sc.s[u >> 2] >> (8u * (u & 3u)) & 0xffu); }
    static __device__ __forceinline__ void unit(const Raw &r, const Scales &sc, uint32_t u, uint32_t, u32x4 &high, u32x4 &low) {
        const uint32_t s = __builtin_amdgcn_perm(0u, sc.s[u >> 2], 0x0c000c00u + 0x00010001u * (u & 3u));  // in both 16-bit halves
        const uint32_t a = (s >> 3) & 0x00070007u, b = s & 0x00070007u;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t q = ((u & 1u) ? r.q[u >> 1][e] >> 4 : r.q[u >> 1][e]) & 0x0f0f0f0fu;
            high[e] = pk_mul(q, a);
            low[e] = pk_mul(q, b);
        }
    }
};

struct KqQ5 {
    static constexpr int TYPE = 5;
    static constexpr uint32_t BLOCK = 176;
    static constexpr int PLANES = 2, SHIFT = 8;
    static constexpr bool PERMUTED = false;
    static constexpr bool HAS_MIN = true;
    struct Raw {
        u32x4 h;
        u32x4 qh;    // the fifth bits of positions 16 h .. + 15, bit u for unit u
        u32x4 q[4];
    };
    typedef KqQ4::Scales Scales;
    typedef KqQ4::Mins Mins;
    static __device__ __forceinline__ void load(const uint8_t *blk, uint32_t, uint32_t h, uint32_t half, Raw &r) {
        if (half == 0u) {
            r.h = *reinterpret_cast<const u32x4 *>(blk);
            r.qh = *reinterpret_cast<const u32x4 *>(blk + 16u + 16u * h);
        }
#pragma unroll
        for (uint32_t c = 2u * half; c < 2u * half + 2u; c++) r.q[c] = *reinterpret_cast<const u32x4 *>(blk + 48u + 32u * c + 16u * h);
    }
    static __device__ __forceinline__ void factors(const Raw &r, float &d, float &dmin, Mins &mins) { KqQ4::header(r.h, d, dmin, mins); }
    static __device__ __forceinline__ Scales prepare(const Raw &r) { return KqQ4::scales(r.h); }
    static __device__ __forceinline__ u32x4 plain(const Raw &r, uint32_t u) {
        return (((u & 1u) ? r.q[u >> 1] >> 4 : r.q[u >> 1]) & 0x0f0f0f0fu) | (((r.qh >> u) & 0x01010101u) << 4);
    }
    static __device__ __forceinline__ int scale(const Scales &sc, uint32_t u) { return KqQ4::scale(sc, u); }
    static __device__ __forceinline__ void unit(const Raw &r, const Scales &sc, uint32_t u, uint32_t, u32x4 &high, u32x4 &low) {
        const uint32_t s = __builtin_amdgcn_perm(0u, sc.s[u >> 2], 0x0c000c00u + 0x00010001u * (u & 3u));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t q = (((u & 1u) ? r.q[u >> 1][e] >> 4 : r.q[u >> 1][e]) & 0x0f0f0f0fu) | (((r.qh[e] >> u) & 0x01010101u) << 4);
            const uint32_t even = pk_mad(q & 0x00ff00ffu, s, 0x00800080u), odd = pk_mad((q >> 8) & 0x00ff00ffu, s, 0x00800080u);
            high[e] = high_bytes(even, odd);
            low[e] = low_bytes(even, odd);
        }
    }
};

struct KqQ6 {
    static constexpr int TYPE = 6;
    static constexpr uint32_t BLOCK = 224;  // padded from 210 at load
    static constexpr int PLANES = 2, SHIFT = 8;
    static constexpr bool PERMUTED = false;
    static constexpr bool HAS_MIN = false;
    struct Raw {
        u32x4 ql[4];  // [2 n + c % 2]: low nibbles unit 4 n + c % 2, high nibbles that + 2
        u32x4 qh[2];  // [n]: bits 2 c of unit 4 n + c
        u32x4 sc;     // sixteen signed scales
        uint32_t d;
    };
    typedef uint32_t Mins;
    struct Scales { uint32_t s[4]; };  // [i]: byte j the scale of the lane's half of unit 2 i + j / 2
    static __device__ __forceinline__ void load(const uint8_t *blk, uint32_t, uint32_t h, uint32_t half, Raw &r) {
        if (half == 0u) {
            r.sc = *reinterpret_cast<const u32x4 *>(blk + 192u);
            r.d = *reinterpret_cast<const uint32_t *>(blk + 208u);
        }
#pragma unroll
        for (uint32_t i = 2u * half; i < 2u * half + 2u; i++) r.ql[i] = *reinterpret_cast<const u32x4 *>(blk + 32u * i + 16u * h);
        r.qh[half] = *reinterpret_cast<const u32x4 *>(blk + 128u + 32u * half + 16u * h);
    }
    static __device__ __forceinline__ void factors(const Raw &r, float &d, float &dmin, Mins &) {
        d = half_bits_to_float(r.d & 0xffffu);
        dmin = 0.f;
    }
    static __device__ __forceinline__ Scales prepare(const Raw &r) {
        Scales s;
#pragma unroll
        for (int i = 0; i < 4; i++) s.s[i] = r.sc[i];
        return s;
    }
    static __device__ __forceinline__ void unit(const Raw &r, const Scales &sc, uint32_t u, uint32_t h, u32x4 &high, u32x4 &low) {
        const uint32_t n = u >> 2, c = u & 3u;
        // Scale 2 u + h, signed, in both 16-bit halves.
        const int one = (int)(sc.s[u >> 1] << (24u - 16u * (u & 1u) - 8u * h)) >> 24;
        const uint32_t s = __builtin_amdgcn_perm(0u, (uint32_t)one, 0x01000100u);
        const uint32_t offset = pk_mad(s, 0xffe0ffe0u, 0x00800080u);  // 128 - 32 s
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t q = ((r.ql[2u * n + (c & 1u)][e] >> (4u * (c >> 1))) & 0x0f0f0f0fu) | (((r.qh[n][e] >> (2u * c)) & 0x03030303u) << 4);
            const uint32_t even = pk_mad(q & 0x00ff00ffu, s, offset), odd = pk_mad((q >> 8) & 0x00ff00ffu, s, offset);
            high[e] = high_bytes(even, odd);
            low[e] = low_bytes(even, odd);
        }
    }
};

struct KqQ3 {
    static constexpr int TYPE = 3;
    static constexpr uint32_t BLOCK = 128;  // repacked at load: eight 16-byte units
    static constexpr int PLANES = 1, SHIFT = 0;
    static constexpr bool PERMUTED = true;
    static constexpr bool HAS_MIN = false;
    struct Raw { u32x4 u[8]; };  // two words of 2-bit values, the high bits, scales - 32 and d
    typedef uint32_t Mins;
    struct Scales {};
    static __device__ __forceinline__ void load(const uint8_t *blk, uint32_t row, uint32_t, uint32_t half, Raw &r) {
#pragma unroll
        for (uint32_t i = 4u * half; i < 4u * half + 4u; i++) r.u[i] = *reinterpret_cast<const u32x4 *>(blk + 16u * (i ^ (row & 7u)));
    }
    static __device__ __forceinline__ void factors(const Raw &r, float &d, float &dmin, Mins &) {
        d = -half_bits_to_float(r.u[0].w >> 16);  // every unit of a block carries the block's d; the planes are negated
        dmin = 0.f;
    }
    static __device__ __forceinline__ Scales prepare(const Raw &) { return Scales{}; }
    static __device__ __forceinline__ void unit(const Raw &r, const Scales &, uint32_t u, uint32_t h, u32x4 &high, u32x4 &) {
        const u32x4 v = r.u[u];
        const int one = (int)(v.w << (24u - 8u * h)) >> 24;
        const uint32_t s = __builtin_amdgcn_perm(0u, (uint32_t)one, 0x01000100u);
        // s * (4 - q) for q = 0 .. 7: the products' low bytes, two of them a multiply.
        const uint32_t p42 = pk_mul(s, 0x00020004u), p31 = pk_mul(s, 0x00010003u), p02 = pk_mul(s, 0xfffe0000u), p13 = pk_mul(s, 0xfffdffffu);
        const uint32_t t0 = __builtin_amdgcn_perm(p31, p42, 0x06020400u), t1 = __builtin_amdgcn_perm(p13, p02, 0x06020400u);
        // Position 4 e + i: bits 2 (e % 4) of byte i of word e / 4, high bit 8 i + e.
        const uint32_t l = h ? v.y : v.x, hb = v.z >> (4u * h);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t q = ((l >> (2 * e)) & 0x03030303u) | (((hb >> e) & 0x01010101u) << 2);
            high[e] = __builtin_amdgcn_perm(t1, t0, q);
        }
    }
};

template <class P> constexpr uint32_t wslot_bytes() { return (32u * (P::BLOCK / 16u) + 63u) / 64u * 1024u; }
template <class P, int RW, int S> constexpr uint32_t lds_bytes() { return S * part_bytes<P>() + S * RW * wslot_bytes<P>(); }
// (the exchange of the parts' sums reuses the rings: 4 RW owners x 3 senders x NT KB)
static_assert(4 * part_bytes<KqQ6>() >= 4 * 2 * 3 * 4 * 1024, "the exchange must fit the token rings");
static_assert(lds_bytes<KqQ3, 4, 2>() >= 4 * 2 * 2 * 2 * 8 * 256 && lds_bytes<KqQ3, 2, 2>() >= 2 * 2 * 2 * 2 * 8 * 256, "nor may the one of two halves' pass the end");
static_assert(lds_bytes<KqQ6, 2, 4>() <= 160 * 1024 && lds_bytes<KqQ5, 2, 4>() <= 160 * 1024, "rings and slots must fit the CU's LDS");

template <class P, int NT, int RW, int S>
__global__ __launch_bounds__(64 * S * RW) __attribute__((amdgpu_waves_per_eu(NT == 4 && P::PLANES == 2 ? 2 : 1))) void matmul_kquant_i8_parts_kernel(
    const uint8_t *qx, const uint8_t *w, const uint8_t *dx, uint32_t k, uint32_t row_bytes, uint32_t qx_bytes, uint32_t w_bytes, uint32_t dx_bytes, uint32_t die_columns, uint32_t die_rows,
    float *out, uint32_t rows, uint32_t n, uint32_t col0, uint32_t out_stride, uint32_t accumulate) {
    // (no struct, and what the first loads need ahead of the rest: the first fourteen words are in registers when the wave starts. A
    // 64-token step over eight layers of 4096 x 14336, quantize_q8 included: 725 -> 700 us.)
    const KqArgs a{qx, w, dx, out, rows, n, k, col0, out_stride, accumulate, row_bytes, qx_bytes, w_bytes, dx_bytes, die_rows};
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr uint32_t CPR = P::BLOCK / 16u, WLOADS = (32u * CPR + 63u) / 64u, WSLOT = wslot_bytes<P>(), XLOADS = 8 / RW;
    constexpr int T = XLOADS + 1;  // loads a wave issues for a token tile
    constexpr bool UNIT_SCALES = NT == 1 && P::HAS_MIN;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, lrow = lane & 31u, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = wave % S, group = wave / S;
    // The chip deals workgroups out to its eight dies in turn. Renumbered, those of a column of the matrix follow one
    // another on one die, whose L2 then has the column's weights for all but the first of them.
    uint32_t column = blockIdx.x, tokens = blockIdx.y;
    if (S <= 2 && die_rows) {
        const uint32_t id = tokens * die_columns + column, dealt = (die_columns & ~7u) * die_rows, turn = id >> 3;
        column = id < dealt ? (turn / die_rows << 3) + (id & 7u) : id / die_rows;
        tokens = (id < dealt ? turn : id) % die_rows;
    }
    const uint32_t n0 = column * (32u * RW) + 32u * group, t0 = tokens * (32u * NT);
    const uint32_t blocks = a.k / 256u, first = part * blocks / S, mine = (part + 1u) * blocks / S - first;
    const uint32_t most = (blocks + S - 1u) / S;  // of any part
    const __amdgpu_buffer_rsrc_t xbuf = make_buffer(a.qx, a.qx_bytes), wbuf = make_buffer(a.w, a.w_bytes), dbuf = make_buffer(a.dx, a.dx_bytes);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
    const uint32_t ring = part * part_bytes<P>(), slot = S * part_bytes<P>() + wave * WSLOT;

    // A step's loads: the tile after the next and its scales, and at a block's first tile the next
    // block's weights (both waves of a part ask for those, the same bytes). A block past the
    // part's last is asked for like the rest, so that every wait counts the same loads, but from
    // where nothing is (an offset with kNowhere's bits set is past any binding): it lands as zeros
    // and adds nothing.
    const uint32_t xlane = (t0 + 8u * (lane >> 4)) * a.k + 16u * ((lane & 15u) ^ (lane >> 4 & 1u));
    const uint32_t dlane = ((t0 + lane) * blocks * 4u) | (lane < 32u ? 0u : kNowhere);
    auto fetch_tile = [&](uint32_t i, uint32_t b, uint32_t tt, uint32_t at, uint32_t dx_at) __attribute__((always_inline)) {
        const uint32_t away = b < mine ? 0u : kNowhere, block = b < mine ? first + b : 0u, run = XLOADS * group + i;
        uint32_t off = i < XLOADS ? xlane : dlane;
        // (Worked out again every time where registers are short: kept, the loads' offsets take sixteen.)
        if (P::HAS_MIN && NT == 4) asm volatile("" : "+v"(off));
        if (i < XLOADS)
            load_lds_b128(xbuf, lds0 + ring + at * TILE_BYTES + RUN * run, (off + (32u * tt + run) * a.k) | away, 256u * block);
        else
            load_lds_b32(dbuf, lds0 + ring + DX_AT + dx_at * DX_BYTES, (off + 32u * tt * blocks * 4u) | away, 4u * block);
    };
    // Chunk c = 64 i + lane of the rows' blocks: row c / CPR, piece c % CPR. A load further is
    // 64 / CPR rows and 64 % CPR pieces further.
    // (Blocks of 128 bytes would meet in the same banks: their pieces are permuted by the row.)
    const uint32_t piece = P::PERMUTED ? (lane % CPR) ^ (lane / CPR & 7u) : lane % CPR;
    const uint32_t wlane = (n0 + lane / CPR) * a.row_bytes + 16u * piece;
    auto fetch_weights = [&](uint32_t i, uint32_t b) __attribute__((always_inline)) {
        const uint32_t away = b < mine ? 0u : kNowhere, block = b < mine ? first + b : 0u;
        const uint32_t pieces = i * (64u % CPR) % CPR, rows = i * (64u / CPR) + i * (64u % CPR) / CPR;
        uint32_t off = wlane;
        if (P::HAS_MIN && NT == 4) asm volatile("" : "+v"(off));
        off += rows * a.row_bytes + 16u * pieces;
        if (pieces > 0u) off += piece + pieces >= CPR ? a.row_bytes - P::BLOCK : 0u;
        if (64u * (i + 1u) > 32u * CPR) off |= lane < 32u * CPR - 64u * i ? 0u : kNowhere;
        load_lds_b128(wbuf, lds0 + slot + 1024u * i, off | away, block * P::BLOCK);
    };

    float acc[NT][16];
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[tt][e] = 0.f;
    // S = 1: the sums of the parts before this one, closed where a part ends. (A row of less than four
    // blocks begins with an empty part, whose sum is a zero; -0 leaves the first part's as they are.) S = 2: the sum
    // of the first of the wave's two parts.
    float closed[S <= 2 ? NT : 1][16];
    if constexpr (S <= 2) {
#pragma unroll
        for (int tt = 0; tt < NT; tt++)
#pragma unroll
            for (int e = 0; e < 16; e++) closed[tt][e] = S == 2 || blocks < 4u ? 0.f : -0.f;
    }
    auto close = [&](int tt) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
            closed[tt][e] += acc[tt][e];
            acc[tt][e] = 0.f;
        }
    };
    uint32_t parts = 1, end = S == 2 ? (2u * part + 1u) * blocks / 4u - first : blocks / 4u;  // S = 1: where the part ends that block b is of; S = 2: where the first ends
    bool closes = false;                    // the block of the last step's tile was its part's last
    u32x4 high[8], low[8];
    i32x16 total = {};  // the last tile's integer sums: finished during the next tile's matrix instructions
    const i32x16 zero = {};
    typename P::Mins mins = {};  // of the block of `total`
    float d = 0.f, dmin = 0.f;
    const uint8_t *const token_at = lds + ring + RUN * (lrow & 7u) + 256u * (lrow >> 3) + 16u * (h ^ (lrow >> 3 & 1u));
    auto sums_at = [&](uint32_t step) __attribute__((always_inline)) { return lds + ring + SUMS_AT + 1024u * (step & 1u) + 16u * lane; };

    // The f32 end of a block over a tile. The lane's sixteen results are tokens 8 j + 4 h + i of its
    // row; element e of them.
    auto finish = [&](float &sum, int e, const f32x16 &msum, const f32x4 &dx) __attribute__((always_inline)) {
        float v = d * (float)total[e];
        if (P::HAS_MIN) v = fmaf(-dmin, msum[e], v);
        sum = fmaf(dx[e & 3], v, sum);
    };
    auto read_dx = [&](uint32_t step, int j) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4 *>(lds + ring + DX_AT + (step & 3u) * DX_BYTES + 32u * j + 16u * h);
    };
    auto minimum_sums = [&](uint32_t step) __attribute__((always_inline)) {
        f32x16 m = {};
        if constexpr (P::HAS_MIN) m = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8 *>(sums_at(step)), mins, m, 0, 0, 0);
        return m;
    };

    auto unit_scale = [](const auto &sc, uint32_t u) __attribute__((always_inline)) {
        if constexpr (P::HAS_MIN) return P::scale(sc, u);
        else return 0;
    };
    // (the first step finishes a tile of zeros)
    *reinterpret_cast<float *>(lds + ring + DX_AT + 3u * DX_BYTES + 4u * lane) = 0.f;
    if (P::HAS_MIN) *reinterpret_cast<u32x4 *>(sums_at(1)) = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (uint32_t i = 0; i < WLOADS; i++) fetch_weights(i, 0);
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)T; i++) fetch_tile(i, 0, 0, 0, 0);
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)T; i++) fetch_tile(i, NT == 1 ? 1 : 0, NT == 1 ? 0 : 1, 1, 1);
    step_end<T, (RW > 1)>();
    uint32_t cur = 0, count = 0;  // the ring's tile of this step; the step's number
    for (uint32_t b = 0; b < most; b++) {
        while (S == 1 && end <= b) end = ++parts * blocks / 4u;
        auto step = [&](auto tile) __attribute__((always_inline)) {
            constexpr int tt = decltype(tile)::value, prev = (tt + NT - 1) % NT;
            const uint32_t ahead = cur == 0u ? 2u : cur - 1u;  // (cur + 2) % 3: last step's
            const uint8_t *tokens = token_at + cur * TILE_BYTES;
            constexpr uint32_t W = tt == 0 ? WLOADS : 0u, L = W + T;
            constexpr uint32_t BEFORE = NT == 1 ? 0u : T;  // tile loads ahead of the weights'
            auto fetch = [&](uint32_t i) __attribute__((always_inline)) {
                if (i >= BEFORE && i < BEFORE + W) fetch_weights(i - BEFORE, b + 1u);
                else fetch_tile(i < BEFORE ? i : i - W, b + (tt + 2) / NT, (tt + 2) % NT, ahead, (count + 2u) & 3u);
            };
            typename P::Raw raw;
            typename P::Scales sc;
            i32x4 af = *reinterpret_cast<const i32x4 *>(tokens), next;
            if (tt == 0) {
                P::load(lds + slot + lrow * P::BLOCK, lrow, h, 0, raw);
                if (NT == 1) {
                    P::load(lds + slot + lrow * P::BLOCK, lrow, h, 1, raw);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                sc = P::prepare(raw);
            }
            const f32x16 msum = minimum_sums(count + 1u);
            f32x4 dx = {};
            i32x16 hsum = {}, lsum = {};
            // Where there are minimums: the sums of the tile's tokens over the lane's half of a unit
            // (below 2048, exact in f16), each of a part's waves those of 8 / RW units, for the next step.
            f16x8 sums = {};
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) {
                if (u < 7) next = *reinterpret_cast<const i32x4 *>(tokens + 32u * (u + 1u));
                if (u % 2 == 0) dx = read_dx(count + 3u, u / 2);
                // The slot is refilled once this wave's reads of it have returned.
                if (tt == 0 && NT > 1 && u == 2) P::load(lds + slot + lrow * P::BLOCK, lrow, h, 1, raw);
                if (tt == 0 && NT > 1 && u == 4) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if constexpr (UNIT_SCALES) {
                    const i32x16 sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, __builtin_bit_cast(i32x4, P::plain(raw, u)), zero, 0, 0, 0);
                    if (u > 0) {
#pragma unroll
                        for (int e = 0; e < 16; e++) hsum[e] = __mul24(unit_scale(sc, u - 1u), lsum[e]) + hsum[e];
                    }
                    lsum = sum;  // scaled while the next unit's instruction runs
                } else {
                    if (tt == 0) P::unit(raw, sc, u, h, high[u], low[u]);
                    hsum = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, __builtin_bit_cast(i32x4, high[u]), u == 0 ? zero : hsum, 0, 0, 0);
                }
                if (!UNIT_SCALES && P::PLANES == 2) lsum = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, __builtin_bit_cast(i32x4, low[u]), u == 0 ? zero : lsum, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 2; e++) finish(acc[prev][2 * u + e], 2 * u + e, msum, dx);
                if (P::HAS_MIN && u < 8 / RW) {
                    const i32x4 q = *reinterpret_cast<const i32x4 *>(tokens + 32u * (8u / RW * group + u));
                    int sum = 0;
#pragma unroll
                    for (int e = 0; e < 4; e++) sum = __builtin_amdgcn_sdot4(q[e], 0x01010101, sum, false);
                    sums[u] = (_Float16)(int16_t)sum;
                }
                // One or two loads a unit: a wave that issues them together stalls until the memory
                // pipeline has taken them, with its matrix instructions behind them.
#pragma unroll
                for (uint32_t i = W > 0u && NT > 1 ? (u < 4u ? u * T / 4u : T + (u - 4u) * W / 4u) : u * L / 8u; i < (W > 0u && NT > 1 ? (u < 4u ? (u + 1u) * T / 4u : T + (u - 3u) * W / 4u) : (u + 1u) * L / 8u); i++) fetch(i);
                // (one unit's fragment ahead and no more: the registers are spoken for)
                __builtin_amdgcn_sched_barrier(0);
                af = next;
            }
            if (P::HAS_MIN) {
                const u32x4 s4 = __builtin_bit_cast(u32x4, sums);
                if (RW == 1) *reinterpret_cast<u32x4 *>(sums_at(count)) = s4;
                if (RW == 2) *reinterpret_cast<uint2 *>(sums_at(count) + 8u * group) = uint2{s4.x, s4.y};
                if (RW == 4) *reinterpret_cast<uint32_t *>(sums_at(count) + 4u * group) = s4.x;
            }
            if (S <= 2 && closes) close(prev);
            if (S <= 2 && tt == 0) closes = end == b + 1u;
            if (tt == 0) P::factors(raw, d, dmin, mins);
#pragma unroll
            for (int e = 0; e < 16; e++) total[e] = UNIT_SCALES ? __mul24(unit_scale(sc, 7), lsum[e]) + hsum[e] : P::PLANES == 2 ? (int)((uint32_t)hsum[e] << P::SHIFT) + lsum[e] : hsum[e];
            cur = cur == RING - 1u ? 0u : cur + 1u;
            count++;
            // The next step's tile (asked for a step ago) and, at a block's end, the next block's
            // weights have landed; this step's own requests may still be out.
            step_end<(tt == 0 && NT > 1 ? T + (int)WLOADS : T), (RW > 1)>();
        };
        step(std::integral_constant<int, 0>{});
        if constexpr (NT >= 2) step(std::integral_constant<int, 1>{});
        if constexpr (NT == 4) {
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
        }
    }
    {
        const f32x16 msum = minimum_sums(count + 1u);
#pragma unroll
        for (int e = 0; e < 16; e++) finish(acc[NT - 1][e], e, msum, read_dx(count + 3u, e / 4));
        if (S == 1) close(NT - 1);
    }
    step_end<0, true>();  // nothing may still land in LDS during the exchange

    // The parts of a row group meet in LDS: the wave of part p finishes sums 16 NT / S p .. + 16 NT / S - 1 of
    // every lane's 16 NT and hands the rest to their owners (S = 2: of both its parts).
    float *inbox = reinterpret_cast<float *>(lds);
    constexpr uint32_t OWN = 16 * NT / S, SENT = S == 4 ? 3 : 2;
    auto place = [&](uint32_t owner, uint32_t from, int i) __attribute__((always_inline)) {
        return (((owner * RW + group) * SENT + from) * OWN + i) * 64u + lane;
    };
    auto sender = [](uint32_t owner, uint32_t from) __attribute__((always_inline)) { return (from + 3u - owner) & 3u; };
#pragma unroll
    for (int owner = 0; owner < (S > 1 ? S : 0); owner++) {
        if (part == (uint32_t)owner) continue;
#pragma unroll
        for (int i = 0; i < (int)OWN; i++) {
            const int e = (int)OWN * owner + i;
            if (S == 4) inbox[place(owner, sender(owner, part), i)] = acc[e / 16][e % 16];
            if constexpr (S == 2) {
                inbox[place(owner, 0, i)] = closed[e / 16][e % 16];
                inbox[place(owner, 1, i)] = acc[e / 16][e % 16];
            }
        }
    }
    if (S > 1) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    // Sum base + i of the lane: tile (base + i) / 16, token 8 (e / 4) + 4 h + e % 4 of it. The buffer
    // ends with the step's last token (out_stride >= n: the tokens after it begin past its end), and lanes
    // past the last row ask past it.
    const __amdgpu_buffer_rsrc_t obuf = make_buffer(reinterpret_cast<const uint8_t *>(a.out + (size_t)t0 * a.out_stride + a.col0), ((min(a.rows - t0, 32u * NT) - 1u) * a.out_stride + a.n) * 4u);
    const uint32_t j = n0 + lrow, olane = (4u * h * a.out_stride + j) * 4u, beyond = j < a.n ? 0u : kNowhere;
    auto collect = [&](auto quarter) __attribute__((always_inline)) {
        constexpr int Q = decltype(quarter)::value, base = 4 * NT * Q;
        // (kNowhere's bits set last: added to, they would carry out of the word)
        auto offset = [&](int i) __attribute__((always_inline)) { return (olane + (32u * ((base + i) / 16) + 8u * (((base + i) % 16) / 4) + (base + i) % 4) * a.out_stride * 4u) | beyond; };
        float held[4 * NT];
        if (a.accumulate) {  // all of them asked for before the first is waited for
#pragma unroll
            for (int i = 0; i < 4 * NT; i++) held[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(obuf, offset(i), 0, 0));
        }
        float sum[4 * NT];
#pragma unroll
        for (int i = 0; i < 4 * NT; i++) {
            sum[i] = S == 1 ? closed[S == 1 ? (base + i) / 16 : 0][(base + i) % 16] : acc[(base + i) / 16][(base + i) % 16];
            if (S == 4) {
                float v[4];
#pragma unroll
                for (int from = 0; from < 4; from++) v[from] = from == Q ? sum[i] : inbox[place(Q, sender(Q, from), i)];
                sum[i] = ((v[0] + v[1]) + v[2]) + v[3];
            }
            if constexpr (S == 2) {
                const float mine0 = closed[(base + i) / 16][(base + i) % 16], sent0 = inbox[place(Q / 2, 0, base + i - (int)OWN * (Q / 2))], sent1 = inbox[place(Q / 2, 1, base + i - (int)OWN * (Q / 2))];
                sum[i] = Q < 2 ? ((mine0 + sum[i]) + sent0) + sent1 : ((sent0 + sent1) + mine0) + sum[i];
            }
        }
        if (a.accumulate) {
#pragma unroll
            for (int i = 0; i < 4 * NT; i++) sum[i] = held[i] + sum[i];
        }
#pragma unroll
        for (int i = 0; i < 4 * NT; i++) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum[i]), obuf, offset(i), 0, 0);
    };
    if (part == 0u) collect(std::integral_constant<int, 0>{});
    if (part == (S == 4 ? 1u : 0u)) collect(std::integral_constant<int, 1>{});
    if (part == (uint32_t)S / 2u) collect(std::integral_constant<int, 2>{});
    if (part == (uint32_t)S - 1u) collect(std::integral_constant<int, 3>{});
}

template <class P, int NT, int RW, int S>
zhip_result launch_tile(const Dispatch &d, const char *name, const KqArgs &a) {
    constexpr uint32_t bytes = lds_bytes<P, RW, S>();
    if (!lds_opt_in<matmul_kquant_i8_parts_kernel<P, NT, RW, S>, (int)bytes>()) return fail(d, ZHIP_E_GPU, "%s: cannot reserve %u bytes of LDS", name, bytes);
    const dim3 grid((a.n + 32u * RW - 1u) / (32u * RW), (a.rows + 32u * NT - 1u) / (32u * NT));
    hipLaunchKernelGGL((matmul_kquant_i8_parts_kernel<P, NT, RW, S>), grid, dim3(64u * S * RW), bytes, d.stream, a.qx, a.w, a.dx, a.k, a.row_bytes, a.qx_bytes, a.w_bytes, a.dx_bytes, grid.x, a.by_die ? grid.y : 0u, a.out, a.rows, a.n, a.col0, a.out_stride, a.accumulate);
    return check_launch(d, name);
}

// The launch of that number in kKquantLaunches, if the format's costs have it.
template <class P, int I>
zhip_result launch_one(const Dispatch &d, const char *name, const KqArgs &a, int best) {
    constexpr KquantLaunch l = kKquantLaunches[I];
    if constexpr (kquant_costs(P::TYPE).has(I))
        if (best == I) return launch_tile<P, (int)l.tiles, (int)l.groups, (int)l.split>(d, name, a);
    if constexpr (I + 1 < kKquantLaunchCount) return launch_one<P, I + 1>(d, name, a, best);
    return fail(d, ZHIP_E_GPU, "%s: no launch", name);
}

template <class P>
zhip_result launch_format(const Dispatch &d, const char *name, KqArgs a) {
    constexpr KquantCosts c = kquant_costs(P::TYPE);
    const int best = kquant_launch(c, a.rows, a.n, a.k, (uint32_t)d.dev->compute_units);
    // Matrices too large for the dies' L2s, several token tiles: 24576 x 3072 and 28672 x 4096 at 256 ... 512 tokens 1 - 8 % faster
    // column by column (two token tiles and one; four the same), matrices of up to 20 MB up to 4 % slower.
    a.by_die = (uint64_t)a.n * a.row_bytes >= (24u << 20);
    return launch_one<P, 0>(d, name, a, best);
}

}  // namespace

// Whole, unsliced k in 256-weight blocks; the caller has validated the bindings and that 32-bit
// offsets reach every operand up to a tile past the last token and row (n + 128 rows, rows + 128
// tokens), and the outputs of 128 tokens, and passes a stride of n or more.
zhip_result launch_matmul_kquant_i8(const Dispatch &d, const char *name, int type, const uint8_t *qx, const uint8_t *w, const uint8_t *dx, float *out,
    uint32_t rows, uint32_t n, uint32_t k, uint32_t col0, uint32_t out_stride, uint32_t accumulate, uint32_t row_bytes, uint32_t qx_bytes, uint32_t w_bytes,
    uint32_t dx_bytes) {
    const KqArgs a{qx, w, dx, out, rows, n, k, col0, out_stride, accumulate, row_bytes, qx_bytes, w_bytes, dx_bytes, 0};
    switch (type) {
    case 3: return launch_format<KqQ3>(d, name, a);
    case 4: return launch_format<KqQ4>(d, name, a);
    case 5: return launch_format<KqQ5>(d, name, a);
    default: return launch_format<KqQ6>(d, name, a);
    }
}

}  // namespace zhip
