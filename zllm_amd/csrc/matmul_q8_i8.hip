// matmul_q8_0 (Q8_0 weights, activations rounded to Q8_0 blocks by quantize_q8) for whole
// 128-deep k steps: the kernel the operation takes when k is a multiple of 128 and not sliced.
// Contract as in matmul_int8.hip (src/kernels/matmul_quant.wgsl):
//   out[t][col0 + j] (+)= sum over 32-position units u of dx[t][u] * dw[j][u] * sum_i(qx * qw),
// every unit's integer sum exact.
//
// The work per output and unit is one 32-deep integer dot product (the int8 matrix cores do
// 1024 of them per instruction) and its scaling by dx * dw, which does not factor out of the
// sum over units. A stream of matrix and vector instructions takes the sum of their times here;
// with four waves a SIMD an f32 add or multiply-add takes 1.1 - 1.3 ns of it, an int -> float conversion
// 2.0 ns, v_mfma_i32_32x32x32_i8 14 - 16 ns and v_mfma_f32_32x32x1_2b_f32 28 ns. So:
//  * the scale products are a matrix instruction: v_mfma_f32_32x32x1_2b_f32 (two independent
//    32 x 32 outer products: lanes 0-31 and 32-63 each give a column of row scales and a row of
//    token scales) yields dx * dw for two token tiles, rounded once to f32 like the vector
//    multiply, in the layout of the integer tiles, in two thirds of the multiplies' time;
//  * the integer sums start from the bits of 1.5 * 2^23 (the matrix instruction's addend): the
//    result's bits are then those of the float 1.5 * 2^23 + sum, and one exact f32 subtraction
//    replaces the conversion.
// Two full-rate vector operations per output and unit remain: 60 ns a unit and 32 x 32 tile in
// registers alone, of the 100 ns that large steps take with their loads, reads and barriers.
// Short steps are bound by the launch, the trips to memory and the exchange at the end.
//
// A workgroup computes 64 (or 32) tokens x 64 matrix rows; wave w multiplies rows 32 (w % 2) .. + 31
// by all the tile's tokens over unit w / 2 of every 128-deep step, lane l holding row (token) l % 32 and bytes
// 16 (l / 32) .. + 15 of the unit. Operands arrive straight in LDS (range-checked buffers: what lies
// past a binding reads as zero) three steps ahead, every wave issuing its share. The scales arrive
// four steps at a time: a step's alone are 8 and 16 bytes of a line a row and token, and a step that
// asked for them moved as many lines for its scales as for its operands, which made it 0.57 us long whatever
// the tile (64 x 4096 x 4096 18.8 -> 13.8 us, 512 x 3072 x 1024 11.8 -> 10.9). At most 128 registers
// a wave and 80 KB a workgroup, so that two workgroups share a CU and one multiplies while the
// other starts or exchanges (512 x 1024 x 6144 22.3 -> 17.1 us, 512 x 4096 x 4096 35.0 -> 31.6; a
// workgroup of 128 tokens and sixteen waves a CU: 20.9, 31.6). The four units'
// sums meet through LDS at the end, always as (u0 + u2) + (u1 + u3): a token's bits depend
// neither on the tokens beside it nor on the tile height.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "round_q8.h"

namespace zhip {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int BN = 64, BK = 128, WAVES = 8, THREADS = 64 * WAVES;
// A step in LDS: token lines [token][128 B], then weight lines [row][128 B]; four steps in the ring.
// The scales come four steps (sixteen units) at a time: [token][16 f32], then [row][16 f16], twice.
constexpr int RING = 4, WBUF = BN * 128, SBUF = BN * 32;
template <int TW>
struct Tile {
    static constexpr int BM = 32 * TW, ABUF = BM * 128, BUF = ABUF + WBUF, DBUF = BM * 64, CHUNK = DBUF + SBUF;
    // The rings, or the exchange of the four units' sums that reuses them (8 waves x 3 inboxes x TW KB).
    static constexpr int RINGS = RING * BUF + 2 * CHUNK, EXCHANGE = WAVES * 3 * TW * 1024, LDS = RINGS > EXCHANGE ? RINGS : EXCHANGE;
    static_assert(2 * LDS <= 160 * 1024, "two workgroups' buffers must fit the CU's LDS");
    // The finished tile behind the exchange, for its rounding: a token's 64 outputs, and four to keep the tokens' out of one another's banks.
    static constexpr int LINE = 68, DONE = EXCHANGE;
    static_assert(DONE + BM * LINE * 4 <= LDS, "the finished tile must fit behind the exchange");
};

struct Q8I8Args {
    const uint8_t *qx;  // rows x k int8
    const uint8_t *w;   // split rows: k int8 values, k / 32 f16 scales, zero pad to 16 bytes
    const uint8_t *dx;  // rows x k / 32 f32
    float *out;
    uint32_t rows, n, k, col0, out_stride, accumulate, row_bytes;
    uint32_t qx_bytes, w_bytes, dx_bytes;  // bytes the kernel may read behind the pointers
    uint8_t *home_qx, *home_dx;  // not null: qx and dx are a multiply's rounding, and belong there too
    uint8_t *next_qx;            // ROUND: the rounded outputs and their scales
    float *next_dx;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buffer(const uint8_t *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, (int)bytes, 0x00020000);
}
typedef __attribute__((address_space(3))) void *lds_ptr;
// One wave-wide load straight into LDS: lane l's bytes land at dst + size * l. The destination
// reaches the load as a bare number, so that the compiler keeps no dependency between these
// loads and the LDS reads of the same wave (it would wait for every load in flight before each
// read); the barriers order them.
__device__ __forceinline__ void load_lds_b128(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t voff, uint32_t soff) {
    asm volatile("" : "+s"(dst));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void load_lds_b32(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t voff, uint32_t soff) {
    asm volatile("" : "+s"(dst));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)dst, 4, voff, soff, 0, 0);
}
// A workgroup barrier after the wave's LDS reads, leaving its newest loads in flight.
template <int LOADS_LEFT>
__device__ __forceinline__ void sync_keeping_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS_LEFT) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// Chunk c (16 bytes) of line r sits at position c ^ key(r): the 32-line fragment reads then run
// at the LDS's full rate.
__device__ __forceinline__ uint32_t line_key(uint32_t row) { return (row & 7u) ^ ((row >> 3) & 1u); }

// ROUND: what is stored is also rounded for the multiply after the next dispatch, as that dispatch would (RoundedCopy): 1, the outputs; 2,
// silu(gate) * up of outputs j and n / 2 + j, for which a workgroup's tile is 32 gate rows and their 32 up rows.
// A quantize_q8 launch is bound by its start and end, and the SiLU pair's reads 8 bytes a value back. us a step, with the launches of quantize_q8 /
// without those that follow a multiply: 28 layers of 1024 x 3072 at 9 / 64 / 512 tokens 1083 / 1165 / 1729 -> 1031 / 1100 / 1634, eight of 2560 x 9728 at
// 128 tokens 845 -> 812, four of 4096 x 14336 at 512 1661 -> 1631.
template <int TW, int ROUND>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4))) void matmul_q8_i8_kernel(
    const uint8_t *qx, const uint8_t *w_rows, const uint8_t *scales, uint32_t k, uint32_t row_bytes, uint32_t qx_bytes, uint32_t w_bytes, uint32_t dx_bytes, uint32_t skip, Q8I8Args a) {
    // (What the first loads need are parameters of their own, ahead of the struct: those are in registers when the wave starts. A
    // 512-token step over 28 layers of 1024 x 3072, quantize_q8 included: 1835 -> 1755 us. The struct's are on their way meanwhile: as
    // parameters of their own the compiler fetches them where the outputs are stored, 0.5 % slower.)
    a.qx = qx, a.w = w_rows, a.dx = scales, a.k = k, a.row_bytes = row_bytes, a.qx_bytes = qx_bytes, a.w_bytes = w_bytes, a.dx_bytes = dx_bytes;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef Tile<TW> T;
    constexpr uint32_t BUF = T::BUF, CHUNKS_AT = RING * BUF, CHUNK = T::CHUNK;
    constexpr int PAIRS = (TW + 1) / 2;
    // Lines a wave loads a step, of tokens and of rows; token lines of a scale load; loads a step and a chunk.
    constexpr uint32_t XROWS = T::BM / WAVES, WROWS = BN / WAVES;
    constexpr int PER_STEP = 2, DL = XROWS / 4, PER_CHUNK = DL + 1;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The tile's rows 0 .. 31 are the matrix's from j0 on, its rows 32 .. 63 `skip` further than that.
    const uint32_t j0 = blockIdx.x * (ROUND == 2 ? BN / 2u : BN), t0 = blockIdx.y * T::BM;
    if (ROUND != 2) skip = 0u;
    const uint32_t steps = a.k / BK;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    // ---- this wave's loads: token lines XROWS wave .. (with 32-token tiles half a wave's load), weight
    // lines WROWS wave ..; a chunk's scales of the same lines, a word a lane.
    const __amdgpu_buffer_rsrc_t xbuf = make_buffer(a.qx, a.qx_bytes), wbuf = make_buffer(a.w, a.w_bytes), dbuf = make_buffer(a.dx, a.dx_bytes);
    const uint32_t xrow = XROWS * wave + (lane >> 3);
    const uint32_t xoff = (t0 + xrow) * a.k + 16u * ((lane & 7u) ^ line_key(xrow));
    const uint32_t wrow = WROWS * wave + (lane >> 3);
    const uint32_t first_row = j0 + (wave >= WAVES / 2u ? skip : 0u);  // (of the wave's lines, less their place in the tile)
    const uint32_t woff = (first_row + wrow) * a.row_bytes + 16u * ((lane & 7u) ^ line_key(wrow));
    // (A step past the end of k is asked for like the rest, so that every wait counts the same loads,
    // but as the last one: nothing reads it.)
    auto fetch = [&](uint32_t buf, uint32_t step) __attribute__((always_inline)) {
        const uint32_t base = lds0 + buf * BUF, at = 128u * min(step, steps - 1u);
        if (XROWS == 8u || lane < 8u * XROWS) load_lds_b128(xbuf, base + 128u * XROWS * wave, xoff, at);
        load_lds_b128(wbuf, base + T::ABUF + 128u * WROWS * wave, woff, at);
    };
    // Units 4 p .. + 3 of token t lie at position p ^ (t / 4 % 4) of its 64 bytes: a step's reads of
    // sixteen tokens fall in sixteen bank groups. (What a ragged last chunk asks for past the end of
    // k is the next row's, or past the buffer's end and zero; nothing reads it. The lanes' offsets
    // are worked out again every time: kept, they would not fit the registers.)
    auto fetch_scales = [&](uint32_t parity, uint32_t chunk) __attribute__((always_inline)) {
        const uint32_t base = lds0 + CHUNKS_AT + parity * CHUNK;
        uint32_t l = lane;
        asm volatile("" : "+v"(l));
        const uint32_t first = (t0 + XROWS * wave + (l >> 4)) * (a.k / 8u) + 64u * chunk;
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)DL; i++)
            load_lds_b32(dbuf, base + 64u * (XROWS * wave + 4u * i), first + i * (a.k / 2u) + 4u * ((l & 15u) ^ (4u * ((XROWS / 4u * wave + i) & 3u))), 0);
        load_lds_b32(wbuf, base + T::DBUF + 32u * WROWS * wave, (first_row + WROWS * wave + (l >> 3)) * a.row_bytes + a.k + 32u * chunk + 4u * (l & 7u), 0);
    };

    // ---- this wave's fragments: rows 32 wn .. + 31, the TW token tiles, unit kq of a step
    const uint32_t lrow = lane & 31u, h = lane >> 5, wn = wave & 1u, kq = wave >> 1;
    const uint32_t chunk = 16u * ((2u * kq + h) ^ line_key(lrow));
    const uint32_t a_at = lrow * 128u + chunk;
    const uint32_t w_at = T::ABUF + (32u * wn + lrow) * 128u + chunk;
    const uint32_t s_at = CHUNKS_AT + T::DBUF + 32u * (32u * wn + lrow) + 2u * kq;
    const uint32_t d_at = CHUNKS_AT + 64u * ((TW == 1 ? 0u : 32u * h) + lrow) + 4u * kq, d_key = 16u * (lrow >> 2 & 3u);

    float acc[TW][16];
#pragma unroll
    for (int i = 0; i < TW; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][e] = 0.f;

    i32x4 w, tok[TW];    // the row's and each tile's token's sixteen bytes of the unit
    float dw, dx[PAIRS];  // the row's scale; the scale of the lane's token in tile 2 pair + lane / 32
    // The operands of the step in buffer `buf` of the ring, its scales those of the chunk at `at`.
    auto read_step = [&](uint32_t buf, uint32_t at) __attribute__((always_inline)) {
        w = *reinterpret_cast<const i32x4 *>(lds + buf * BUF + w_at);
        dw = (float)*reinterpret_cast<const _Float16 *>(lds + at + s_at + 8u * buf);
#pragma unroll
        for (int tt = 0; tt < TW; tt++) tok[tt] = *reinterpret_cast<const i32x4 *>(lds + buf * BUF + a_at + 4096 * tt);
#pragma unroll
        for (int pair = 0; pair < PAIRS; pair++) dx[pair] = *reinterpret_cast<const float *>(lds + at + (d_at + ((16u * buf) ^ d_key)) + 4096 * pair);
    };
    // The integer sums start from the bits of 1.5 * 2^23: bits + sum are then the bits of the
    // float 1.5 * 2^23 + sum (|sum| <= 32 * 127 * 127 < 2^22, one unit in the last place is 1), and
    // the exact subtraction below replaces a conversion (half the rate of an addition here).
    constexpr int MAGIC_BITS = 0x4B400000;
    constexpr float MAGIC = 12582912.f;
    i32x16 magic;
#pragma unroll
    for (int e = 0; e < 16; e++) magic[e] = MAGIC_BITS;
    asm volatile("" : "+v"(magic));  // sixteen registers, set once
    auto multiply = [&]() __attribute__((always_inline)) {
        const f32x32 none = {};
#pragma unroll
        for (int pair = 0; pair < PAIRS; pair++) {
            i32x16 sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, tok[2 * pair], magic, 0, 0, 0);
            const f32x32 scale = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dx[pair], none, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; e++) acc[2 * pair][e] = fmaf(__int_as_float(sums[e]) - MAGIC, scale[e], acc[2 * pair][e]);
            if (2 * pair + 1 < TW) {
                sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, tok[2 * pair + 1 < TW ? 2 * pair + 1 : 0], magic, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; e++) acc[2 * pair + 1 < TW ? 2 * pair + 1 : 0][e] = fmaf(__int_as_float(sums[e]) - MAGIC, scale[16 + e], acc[2 * pair + 1 < TW ? 2 * pair + 1 : 0][e]);
            }
        }
    };

    fetch_scales(0, 0);
    fetch(0, 0);
    fetch(1, 1);
    fetch(2, 2);
    sync_keeping_loads<2 * PER_STEP>();  // the first scales and step 0 have landed

    // Step s multiplies buffer s % 4 while buffer (s + 3) % 4 is refilled. A chunk's first step asks for
    // the next chunk's scales.
    uint32_t at = 0;  // the chunk of step s's scales
    auto step = [&](uint32_t s, auto phase) __attribute__((always_inline)) {
        constexpr uint32_t p = decltype(phase)::value;
        read_step(p, at);
        if (p == 0) fetch_scales(at == 0u ? 1u : 0u, s / 4u + 1u);
        fetch((p + 3u) & 3u, s + 3u);
        if (p == 3) at = at == 0u ? CHUNK : 0u;
        multiply();
        // (Nothing of a step's scaling may be left for later: its operands would pile up in registers.)
#pragma unroll
        for (int i = 0; i < TW; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) asm volatile("" : "+v"(acc[i][e]));
        sync_keeping_loads<2 * PER_STEP + (p < 2 ? PER_CHUNK : 0)>();  // step s + 1 has landed; buffer s % 4 has been read
    };
    uint32_t s = 0;
    for (; s + 4u <= steps; s += 4u) {
        step(s, std::integral_constant<uint32_t, 0>{});
        step(s + 1u, std::integral_constant<uint32_t, 1>{});
        step(s + 2u, std::integral_constant<uint32_t, 2>{});
        step(s + 3u, std::integral_constant<uint32_t, 3>{});
    }
    if (s < steps) step(s, std::integral_constant<uint32_t, 0>{});
    if (s + 1u < steps) step(s + 1u, std::integral_constant<uint32_t, 1>{});
    if (s + 2u < steps) step(s + 2u, std::integral_constant<uint32_t, 2>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still land in LDS during the exchange
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    // The rounding this launch reads, to where the caller has it: sixteen bytes a thread, the first on their way during the exchange.
    const uint32_t pieces = a.home_qx ? (a.qx_bytes + a.dx_bytes) / 16u : 0u, values = a.qx_bytes / 16u;
    const uint32_t piece0 = a.home_qx ? (blockIdx.y * gridDim.x + blockIdx.x) * THREADS + tid : 0u;
    auto piece = [&](uint32_t i) __attribute__((always_inline)) { return i < values ? reinterpret_cast<const uint4 *>(a.qx)[i] : reinterpret_cast<const uint4 *>(a.dx)[i - values]; };
    auto settle = [&](uint32_t i, const uint4 &v) __attribute__((always_inline)) { (i < values ? reinterpret_cast<uint4 *>(a.home_qx)[i] : reinterpret_cast<uint4 *>(a.home_dx)[i - values]) = v; };
    uint4 moved = {};
    if (piece0 < pieces) moved = piece(piece0);

    // The four units of a tile meet in LDS: a row half's 4 TW quarters of tiles (quarter p of tile tt: the
    // lane's sums 4 p .. + 3) are shared out, quarter i to the wave of unit i / TW, and each wave hands the
    // others' to their owners.
    f32x4 *inbox = reinterpret_cast<f32x4 *>(lds);
    auto slot = [&](uint32_t owner, uint32_t from, int i) {
        return (((owner * 2u + wn) * 3u + ((from + 3u - owner) & 3u)) * TW + i) * 64u + lane;
    };
    auto mine = [&](int i) { return f32x4{acc[i / 4][4 * (i % 4)], acc[i / 4][4 * (i % 4) + 1], acc[i / 4][4 * (i % 4) + 2], acc[i / 4][4 * (i % 4) + 3]}; };
    auto send = [&](auto quarter) __attribute__((always_inline)) {
        constexpr int Q = decltype(quarter)::value;
#pragma unroll
        for (int i = 0; i < 4 * TW; i++)
            if (i / TW != Q) inbox[slot(i / TW, Q, i % TW)] = mine(i);
    };
    const bool aligned = ((a.out_stride | a.col0) & 3u) == 0u && (reinterpret_cast<uintptr_t>(a.out) & 15u) == 0u;
    // In each 32 x 32 tile the lane holds rows 8 p + 4 (lane / 32) .. + 3, p < 4, of token
    // lane % 32: sixteen contiguous bytes of the token's output row per quarter.
    float *done = reinterpret_cast<float *>(lds + T::DONE);
    auto collect = [&](auto quarter) __attribute__((always_inline)) {
        constexpr int Q = decltype(quarter)::value;
#pragma unroll
        for (int i = Q * TW; i < (Q + 1) * TW; i++) {
            const uint32_t t = t0 + 32u * (i / 4) + lrow, col = j0 + 32u * wn + (wn ? skip : 0u) + 8u * (i % 4) + 4u * h;
            f32x4 part[4];
#pragma unroll
            for (int from = 0; from < 4; from++) part[from] = from == Q ? mine(i) : inbox[slot(Q, from, i % TW)];
            f32x4 v = (part[0] + part[2]) + (part[1] + part[3]);
            if (t >= a.rows || col >= a.n) continue;
            float *o = a.out + (size_t)t * a.out_stride + a.col0 + col;
            if (aligned && col + 3u < a.n) {
                f32x4 *o4 = reinterpret_cast<f32x4 *>(o);
                if (a.accumulate) v += *o4;
                *o4 = v;
                if (ROUND) *reinterpret_cast<f32x4 *>(done + (32u * (i / 4) + lrow) * T::LINE + 32u * wn + 8u * (i % 4) + 4u * h) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (col + r < a.n) o[r] = a.accumulate ? o[r] + v[r] : v[r];
            }
        }
    };
    switch (kq) {
    case 0: send(std::integral_constant<int, 0>{}); break;
    case 1: send(std::integral_constant<int, 1>{}); break;
    case 2: send(std::integral_constant<int, 2>{}); break;
    default: send(std::integral_constant<int, 3>{}); break;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    switch (kq) {
    case 0: collect(std::integral_constant<int, 0>{}); break;
    case 1: collect(std::integral_constant<int, 1>{}); break;
    case 2: collect(std::integral_constant<int, 2>{}); break;
    default: collect(std::integral_constant<int, 3>{}); break;
    }
    if (piece0 < pieces) settle(piece0, moved);
    if (pieces > THREADS * gridDim.x * gridDim.y)
        for (uint32_t i = piece0 + THREADS * gridDim.x * gridDim.y; i < pieces; i += THREADS * gridDim.x * gridDim.y) settle(i, piece(i));

    // Eight lanes a 32-value block, four values each, as quantize_q8 has them.
    if constexpr (ROUND != 0) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        constexpr uint32_t LANES = ROUND == 2 ? 8u : 16u;  // a token
        const uint32_t width = ROUND == 2 ? a.n / 2u : a.n;
#pragma unroll
        for (uint32_t i = 0; i < (T::BM * LANES + THREADS - 1u) / THREADS; i++) {
            const uint32_t at = tid + THREADS * i, token = at / LANES, c = 4u * (at % LANES);
            if (T::BM * LANES % THREADS != 0u && at >= T::BM * LANES) break;  // (whole waves)
            const qf32x4 *line = reinterpret_cast<const qf32x4 *>(done + token * T::LINE + c);
            qf32x4 v = line[0];
            if (ROUND == 2) v = silu_pair(v, line[8]);
            float mag = fabsf(v[0]);
#pragma unroll
            for (int e = 1; e < 4; e++) mag = fabsf(v[e]) > mag ? fabsf(v[e]) : mag;
            int q[4];
            const float d = round_block(v, max_of_eight(mag), q);
            if (t0 + token >= a.rows || j0 + c >= width) continue;
            const size_t to = (size_t)(t0 + token) * width + j0 + c;
            reinterpret_cast<uint32_t *>(a.next_qx)[to / 4u] = four_bytes(q);
            if (at % 8u == 0u) a.next_dx[to / 32u] = d;
        }
    }
}

template <int TW, int ROUND>
zhip_result launch_tile(const Dispatch &d, const char *name, const Q8I8Args &a) {
    typedef Tile<TW> T;
    if (!lds_opt_in<matmul_q8_i8_kernel<TW, ROUND>, T::LDS>()) return fail(d, ZHIP_E_GPU, "%s: cannot reserve %d bytes of LDS", name, T::LDS);
    const dim3 grid((a.n + BN - 1) / BN, (a.rows + T::BM - 1) / T::BM);
    hipLaunchKernelGGL((matmul_q8_i8_kernel<TW, ROUND>), grid, dim3(THREADS), T::LDS, d.stream, a.qx, a.w, a.dx, a.k, a.row_bytes, a.qx_bytes, a.w_bytes, a.dx_bytes, a.n / 2u - BN / 2u, a);
    return check_launch(d, name);
}
template <int TW>
zhip_result launch_round(const Dispatch &d, const char *name, const Q8I8Args &a, uint32_t round) {
    return round == 0u ? launch_tile<TW, 0>(d, name, a) : round == 1u ? launch_tile<TW, 1>(d, name, a) : launch_tile<TW, 2>(d, name, a);
}

}  // namespace

// Whole, unsliced k in 128-deep steps (the caller has validated the bindings and that 32-bit
// offsets reach a tile past the operands' ends).
bool matmul_q8_i8_accepts(uint32_t k, uint32_t k_slice, uint32_t slices) { return slices == 1u && k_slice >= k && k >= BK && k % BK == 0u; }

zhip_result launch_matmul_q8_i8(const Dispatch &d, const char *name, const uint8_t *qx, const uint8_t *w, const uint8_t *dx, float *out, uint32_t rows,
    uint32_t n, uint32_t k, uint32_t col0, uint32_t out_stride, uint32_t accumulate, uint32_t row_bytes, uint32_t qx_bytes, uint32_t w_bytes,
    uint32_t dx_bytes) {
    Q8I8Args a{};
    a.qx = qx; a.w = w; a.dx = dx; a.out = out;
    a.rows = rows; a.n = n; a.k = k; a.col0 = col0; a.out_stride = out_stride; a.accumulate = accumulate;
    a.row_bytes = row_bytes; a.qx_bytes = qx_bytes; a.w_bytes = w_bytes; a.dx_bytes = dx_bytes;
    if (d.rounded_in && d.rounded_in->data && d.rounded_in->q == qx && d.rounded_in->d == dx && d.rounded_in->rows == rows && d.rounded_in->k == k) {
        a.home_qx = d.rounded_in->q; a.home_dx = d.rounded_in->d;
        a.qx = d.rounded_in->data; a.dx = a.qx + d.rounded_in->scales_at();
    }
    uint32_t round = 0;
    RoundedCopy *next = d.rounded_out;
    if (next && next->x == out && next->rows == rows && col0 == 0u && out_stride == n && n == (next->mode == 2u ? 2u * next->k : next->k) && (reinterpret_cast<uintptr_t>(out) & 15u) == 0u) {
        if (uint8_t *to = next->reserve(d)) {
            round = next->mode == 2u ? 2u : 1u;
            a.next_qx = to; a.next_dx = reinterpret_cast<float *>(to + next->scales_at());
        }
    }
    // The tile whose workgroups, two a CU, take least: costs fitted to both tiles' times at 16 ... 512 tokens over sixteen
    // matrices of 1024 x 3072 ... 28672 x 4096, where the rule's tile is the faster one but for 0.01 % of the time in the mean (64-token tiles
    // wherever they kept half of the CUs busy, as here before, 0.6 %). us, 64 / 32: 512 x 1024 x 2048 (256 workgroups of 64
    // tokens) 7.9 / 8.3, 201 x 2560 x 4096 (256) 13.8 / 15.1, 512 x 28672 x 4096 203 / 287; 80 x 5120 x 2560 (160) 12.9 / 10.1, 160 x
    // 3072 x 1024 (144) 7.2 / 5.6, 512 x 2048 x 1024 (128) 10.7 / 8.6, 64 x 4096 x 4096 (64) 18.0 / 13.8.
    constexpr SharedCu tall{52, 85}, flat{40, 60};
    const uint64_t columns = (n + BN - 1) / BN, cus = (uint64_t)d.dev->compute_units;
    const zhip_result r = tall.of((rows + 63u) / 64u * columns, cus) < flat.of((rows + 31u) / 32u * columns, cus) ? launch_round<2>(d, name, a, round) : launch_round<1>(d, name, a, round);
    if (r == ZHIP_OK && round != 0u) next->data = a.next_qx;
    return r;
}

}  // namespace zhip
