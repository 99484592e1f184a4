// matvec_bf16 (and matvec_f16) on the matrix cores for steps of several tokens and k = 1024 ... 4096 in steps of
// 512: the weight stream is read once for all tokens of the step and nothing but partial sums
// crosses LDS. (Rows of more than 4096 weights and no multiple of 512 are taken as if they ended in zeros: their lines are
// whole, the ones past a row's end are asked for from an empty buffer, and the tokens' positions there are zeros.) Contract of src/kernels/matvec_half.wgsl:1-133 with the bf16 decoder of
// src/kernels/half/bf16.wgsl:3-9: out[t][col0 + j] (+)= sum_i x[t][i] * w[j][i], the inputs
// taken as the f32 values they are. (The reference gives every token a row of workgroups of its
// own, so a step of M tokens reads the weights M times.)
//
// Arithmetic. v_mfma_f32_32x32x16_bf16 multiplies 32 rows of inputs by 32 weight rows over
// sixteen positions. The weights are bf16 already and reach the instruction as loaded. An f32
// input is the exact sum of three bf16 values (f16 weights have their own split, see F16 below;
// of bf16: its upper sixteen bits, the upper sixteen bits of
// what that left, and the rest: eight significant bits each), so a token enters as three operand
// rows, every product is exact in the f32 accumulator, and the three rows' sums are added at the
// end. Eight tokens fill 24 of the 32 operand rows; the other eight are zeros. A token's rows
// meet no other token's anywhere: its results do not depend on how many tokens share the launch
// (steps of more than eight tokens run as launches of eight). Sums stay short: a piece of 64 positions
// (below) is four instructions' chain, a wave adds its pieces' sums, and the eight waves' meet in
// pairs. (One chain over a wave's pieces and one over the waves had up to 1.3 times the general
// kernel's error, gate / up steps of 4096 weights a row at eight tokens 2.36e-7 in bf16 and 2.55e-7 in
// f16; now 1.76e-7 and 1.84e-7 beside 1.94e-7. In time it shows nowhere.)
//
// Layout of the work. A 512-thread workgroup is eight waves that split k eight ways; a wave
// builds its k range of all tokens' operand rows once, into registers (k / 32 VGPRs), from the pieces that
// the workgroup has put in LDS, a wave a token, or that a launch in front has left in memory. Persistent
// workgroups take 32-row weight tiles b, b + G, ... and at the end a share of the rows left
// over, in units of eight rows, so that every workgroup reads the same number of bytes within
// one unit. A wave's part of a tile is k / 512 pieces, a piece one 128-byte line (64 positions)
// of each of the 32 rows; pieces arrive in a private ring of 4 KB LDS slots by wave-wide direct
// loads of whole lines (lane l of load j brings 16 bytes of row 8 j + l / 8), two pieces
// ahead of the one multiplied, and each lane reads its row's sixteen bytes of a sixteen-position
// step back for one matrix instruction. (The matrix instruction wants lane l to hold row l % 32:
// a lane loading its own bytes would make every lane of a load touch another cache line, and the
// vector memory unit moves sixteen bytes per line it looks up.) Chunk c (16 bytes) of row r sits
// at position c ^ (r / 2 % 8) of the row's line in the slot: two neighbouring lines fill the 64
// banks once, and sixteen rows' reads of one chunk fall in sixteen different groups of four. The eight waves' partial sums meet in LDS, where
// 256 threads add the eight for one output each, neighbouring k ranges first; the outputs wait
// in LDS and are stored when the workgroup's run ends (or every 40 tiles), 128 contiguous bytes
// a token and tile. One barrier a tile; no barrier waits for the loads in flight.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "decode.h"
#include "matvec_common.h"

namespace zhip {

namespace {

typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 hf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 hf16x4 __attribute__((ext_vector_type(4)));
typedef float hf32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t hu32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t THREADS = 512, WAVES = 8;
constexpr int DEPTH = 3;  // ring slots a wave: two pieces in flight behind the one multiplied (four measured no faster)
constexpr int LOADS = 4;  // wave-wide loads a piece: eight rows each
constexpr uint32_t SLOT = 32u * 128u;
constexpr uint32_t PART_BYTES = 2u * WAVES * 256u * 4u;  // [tile parity][wave][token of the lane's four][lane]
constexpr uint32_t KEPT = 40;                            // tiles whose outputs wait in LDS for one burst of stores
constexpr uint32_t RING_BYTES = WAVES * DEPTH * SLOT;
constexpr uint32_t LDS_BYTES = PART_BYTES + RING_BYTES + KEPT * 1024u + 64u;  // (the last 64: f16 tokens' inverse scales)
// Kernels whose workgroups split their tokens themselves keep the pieces in LDS ([piece][token of
// 8][k], rows padded by 16 bytes so that one chunk of neighbouring rows falls in different banks)
// until the operands are read, at its end: ring slots below them take their weights meanwhile.
// An f16 token enters as two pieces, `whole` (steps of a pair, and over some long rows) as three, and so does every other.
constexpr uint32_t pieces_of(bool f16, bool whole) { return f16 && !whole ? 2u : 3u; }
template <int NP> constexpr uint32_t piece_row() { return 1024u * NP + 16u; }
template <int NP, uint32_t PIECES> constexpr uint32_t pieces_bytes() { return 8u * PIECES * piece_row<NP>(); }
template <int NP, uint32_t PIECES> constexpr bool pieces_fit() { return pieces_bytes<NP, PIECES>() <= LDS_BYTES - 64u; }
static_assert(LDS_BYTES <= 160u * 1024u - 64u, "the rings must fit the CU's LDS");

struct StreamArgs {
    MvArgs a;
    uint32_t w_bytes;    // bytes of the weights the loads may touch (they are range-checked)
    uint32_t rounds;     // 32-row tiles every workgroup takes: tiles b, b + G, ...
    uint32_t tail_base;  // units of eight rows after those: tail_base for every workgroup
    uint32_t tail_rem;   // and one more for each of the first tail_rem
    uint32_t by_die;     // workgroups renumbered die by die (the grid is a multiple of eight)
    // Inputs split beforehand (SPLIT kernels): planes [piece][token][k] of the weights' type.
    const uint8_t *planes;
    uint32_t plane_tokens;  // tokens a plane holds
    uint32_t plane_k;       // positions of a token in a plane (the whole row's, of which the launch may take a stretch)
    uint32_t plane_first;   // the launch's first position
    uint32_t t0;            // the launch's first token in the planes
    const float *inverse;   // F16 kernels: one over each token's scale
    // Rows of more than 4096 weights in equal stretches of columns (LONG kernels): `parts`
    // workgroups share a tile, a stretch each, and leave their sums in `partial`
    // ([part][token of 8][output], outputs a.rows apart).
    uint32_t parts;
    float *partial;
};

// A barrier that waits for this wave's LDS traffic only: the weight loads of the pieces ahead
// stay in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A 4-byte store the compiler's wait-count bookkeeping does not see as a store: with one pending
// it would turn every wait for a weight load into a wait for all loads in flight (loads and
// stores complete out of order with each other). A wait that counts only the loads issued
// after the awaited one stays sufficient while a store is outstanding.
__device__ __forceinline__ void store_apart(float *at, float v) {
    asm volatile("global_store_dword %0, %1, off\n\ts_nop 0" ::"v"(at), "v"(v) : "memory");
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buffer(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
typedef __attribute__((address_space(3))) void *lds_ptr;
// One wave-wide load of 16 bytes a lane straight into LDS (lane l lands at dst + 16 l). The
// destination reaches the load as a bare LDS address, so the compiler keeps no dependency
// between these loads and later LDS reads; the explicit waits order them.
__device__ __forceinline__ void load_lds_b128(__amdgpu_buffer_rsrc_t buf, uint32_t dst, uint32_t voffset) {
    asm volatile("" : "+s"(dst));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (lds_ptr)(uintptr_t)dst, 16, voffset, 0, 0, 0);
}
template <int LEFT>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}

// The bits of one of the three pieces of x (the one whose mask is all ones; the others' are
// zero) as an f32 whose lower half is zero: x is the exact sum of the three. Infinities and NaNs stay what they are in the first piece; the others are zero.
__device__ __forceinline__ uint32_t piece_bits(float x, uint32_t m0, uint32_t m1, uint32_t m2) {
    const uint32_t b = __float_as_uint(x);
    const bool finite = (b & 0x7f800000u) != 0x7f800000u;
    // (selects, not branches: a NaN whose payload sits in the lower half would otherwise be cut to an infinity)
    const uint32_t p0 = (b & 0xffff0000u) | ((!finite & ((b & 0x007fffffu) != 0u)) ? 0x00400000u : 0u);
    const float d1 = x - __uint_as_float(p0);
    const float r1 = finite ? d1 : 0.f;
    const uint32_t p1 = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(p1);
    return (p0 & m0) | (p1 & m1) | (__float_as_uint(r2) & m2);
}

// The upper halves of two words as a pair of bf16 values, `lo` first.
__device__ __forceinline__ uint32_t upper_halves(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

// Piece p of four values.
__device__ __forceinline__ uint2 bf16_piece(const float4 &v, uint32_t p) {
    const uint32_t m0 = p == 0u ? ~0u : 0u, m1 = p == 1u ? ~0u : 0u, m2 = p == 2u ? ~0u : 0u;
    uint2 w;
    w.x = upper_halves(piece_bits(v.x, m0, m1, m2), piece_bits(v.y, m0, m1, m2));
    w.y = upper_halves(piece_bits(v.z, m0, m1, m2), piece_bits(v.w, m0, m1, m2));
    return w;
}

// The larger of `big` and the magnitudes in v, infinities left out with FINITE (and NaNs always).
template <bool FINITE>
__device__ __forceinline__ float largest(float big, const float4 &v) {
    const float x[4] = {fabsf(v.x), fabsf(v.y), fabsf(v.z), fabsf(v.w)};
#pragma unroll
    for (int j = 0; j < 4; j++) big = fmaxf(big, FINITE && x[j] == __builtin_inff() ? 0.f : x[j]);
    return big;
}

// The power of two that puts a token's largest finite magnitude `big` in [2^14, 2^15) (2^126 for one
// below the normal numbers), and one over it.
__device__ __forceinline__ void f16_scale(float big, float &scale, float &inverse) {
    const int e = (int)((__float_as_uint(big) >> 23) & 0xffu);  // biased exponent; 0 for zero and subnormals
    int se = 127 + 14 - (e - 127);                               // scale = 2^(14 - (e - 127)), kept normal both ways
    se = se < 1 ? 1 : se > 253 ? 253 : se;
    scale = __uint_as_float((uint32_t)se << 23);
    inverse = __uint_as_float((uint32_t)(254 - se) << 23);
}

// Four scaled values as their f16 roundings, what those left times 2^11 and, with PIECES 3, what that left
// times 2^22: eleven significant bits each, an f32 input's 24 in three. Infinities and NaNs are what they are
// in the first; what an infinity leaves, a NaN, becomes a finite number, any being as good beside it.
template <uint32_t PIECES>
__device__ __forceinline__ void f16_pieces(const float4 &v, float scale, uint2 (&w)[PIECES]) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    _Float16 q[PIECES][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        // The scale is a power of two, so x * scale - q in one fused operation is exact, and so is what the next leaves.
        q[0][j] = (_Float16)(x[j] * scale);
        const float rest = fmaxf(fmaf(x[j], scale, -(float)q[0][j]) * 2048.0f, -32768.0f);
        q[1][j] = (_Float16)rest;
        if constexpr (PIECES == 3) q[2][j] = (_Float16)((rest - (float)q[1][j]) * 2048.0f);
    }
#pragma unroll
    for (uint32_t p = 0; p < PIECES; p++) w[p] = __builtin_bit_cast(uint2, hf16x4{q[p][0], q[p][1], q[p][2], q[p][3]});
}

// NP: pieces of a wave's k range (k = 512 NP). SPLIT: the tokens' three pieces come ready from
// matvec_bf16_split_kernel's planes (long rows, and where the pieces do not fit LDS). Otherwise
// every workgroup normalises and splits the tokens itself, a wave each, through LDS: 1 us of the
// workgroup's time where a launch in front costs 3 (8 tokens with the RMSNorm prologue: f16 4096 x
// 2048 11.6 -> 8.6 us, 151936 x 1024 56.7 -> 52.9, 4096 x 4096 17.9 -> 13.1; bf16 12.4 -> 8.8,
// 56.1 -> 53.3).
// F16 (matvec_f16: the weights are f16 and the matrix instruction v_mfma_f32_32x32x16_f16): a
// token enters as two f16 rows, the rounding of its inputs and the rounding of what that left
// times 2^11, after a power of two has put its largest magnitude at 2^14 (an input keeps 22
// bits), and a token's sums are multiplied by one over its scale. With PAIR there is a third row,
// what those two left times 2^22, and an input keeps all its bits (the general kernel, which takes
// pairs without ZHIP_OPTION_WIDE_DECODE, has them too): the matrix instruction has the rows anyway. So over the long
// rows that would be the general kernel's otherwise (no multiple of 512, or under 16 MB): an activation's products there, of a log-normal magnitude,
// 768 x 6400, relative error 1.17e-7 with two, 1.08e-7 with three, 1.12e-7 in the general kernel. (In time three cost up to 10 %: 2560 x 9728
// 16.7 -> 18.5 us.)
// PAIR: a SILU_PAIR step, an output tile's gate rows and then its up rows (the general kernel's
// time grows with the tokens: 2 x 8192 x 2048 f16 at eight 38 us, here 18).
// LONG: rows of q.parts stretches of 512 NP columns (the last one may end past the row); workgroup i multiplies stretch i % parts (`kpart`) of the tiles that
// walker i / parts takes, and launch_matvec_parts_sum adds the stretches' sums. Without the RMSNorm prologue no
// workgroup needs more of a token than its stretch (an F16 token's scale is then the stretch's own).
template <int NP, bool SPLIT, bool F16, bool LONG, bool PAIR, bool WHOLE>
__global__ __launch_bounds__(THREADS) void matvec_bf16_mfma_stream_kernel(const float *first_x, const uint8_t *first_w, const float *first_norm_w, uint32_t k_flags, uint32_t xr, uint32_t row_bytes,
    uint32_t rows, uint32_t half_at, uint32_t w_bytes, uint32_t rounds_walkers, uint32_t counts, StreamArgs q) {
    // (what the first loads are addressed by is in registers when the wave starts: see MV_FIRST. Some share a word: launch_blocks)
    q.a.x = first_x, q.a.w = first_w, q.a.norm_w = first_norm_w, q.a.k = k_flags & 0xffffffu, q.a.flags = k_flags >> 24, q.a.xr = xr, q.a.row_bytes = row_bytes, q.a.rows = rows;
    q.a.half = half_at, q.w_bytes = w_bytes, q.rounds = rounds_walkers & 0xffffu, q.tail_rem = counts & 0xffffu, q.tail_base = counts >> 16 & 15u, q.a.m = counts >> 20 & 15u, q.by_die = counts >> 24 & 1u;
    q.parts = counts >> 25;
    static_assert(!PAIR || !LONG, "gate / up steps take whole rows");
    constexpr uint32_t PER = PAIR ? 2u : 1u;  // weight tiles an output tile
    constexpr uint32_t PIECES = pieces_of(F16, WHOLE);
    static_assert(SPLIT || pieces_fit<NP, PIECES>(), "the tokens' pieces must fit LDS");
    const MvArgs &a = q.a;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    float *lds_part = reinterpret_cast<float *>(lds);
    float *lds_kept = reinterpret_cast<float *>(lds + PART_BYTES + RING_BYTES);  // [tile % KEPT][token][row]
    float *lds_inverse = lds_kept + KEPT * 256u;                                 // [token], read behind the tiles' barriers
    if (F16 && SPLIT && threadIdx.x < 8u) lds_inverse[threadIdx.x] = threadIdx.x < a.m ? q.inverse[q.t0 + threadIdx.x] : 1.0f;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *ring = lds + PART_BYTES + wave * SLOT;  // [slot][wave]
    const uint32_t ring0 = (uint32_t)(uintptr_t)ring;
    const __amdgpu_buffer_rsrc_t wbuf = make_buffer(a.w, q.w_bytes), nobuf = make_buffer(a.w, 0);

    // The workgroup's tiles: b, b + G, ... and its share of the rows after the whole rounds. The
    // hardware deals workgroups out to the chip's eight dies in turn; b numbers them so that a
    // die's workgroups take neighbouring tiles (one die then reads a contiguous eighth of every
    // round's stretch of the matrix: 55 us against 58 us for four tokens over 151936 x 1024).
    const uint32_t kpart = LONG ? blockIdx.x % q.parts : 0u, walker = LONG ? blockIdx.x / q.parts : blockIdx.x;
    const uint32_t G = rounds_walkers >> 16;
    const uint32_t b = q.by_die ? (walker & 7u) * (G >> 3) + (walker >> 3) : walker;
    const uint32_t tail_units = q.tail_base + (b < q.tail_rem ? 1u : 0u);
    const uint32_t tail_row = 32u * q.rounds * G + 8u * (b * q.tail_base + (b < q.tail_rem ? b : q.tail_rem));
    const uint32_t count = q.rounds + (tail_units ? 1u : 0u);
    auto first_row = [&](uint32_t o) { return o < q.rounds ? 32u * (b + o * G) : tail_row; };
    auto rows_of = [&](uint32_t o) { return o < q.rounds ? 32u : 8u * tail_units; };

    // A piece's loads: load j brings rows 8 j .. 8 j + 7, lane l row 8 j + l / 8 and the chunk
    // that belongs at position l % 8 of its line. The whole address is the lane's offset, which
    // is what the buffer's range check sees: rows past the matrix's end land as zeros.
    auto line_key = [](uint32_t row) { return (row >> 1) & 7u; };
    uint32_t woff[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; j++) woff[j] = (8u * j + (lane >> 3)) * a.row_bytes + 1024u * NP * kpart + 128u * NP * wave + 16u * ((lane & 7u) ^ line_key(8u * j + (lane >> 3)));
    uint32_t load_tile = 0, load_piece = 0, load_slot = 0;
    auto issue = [&]() __attribute__((always_inline)) {
        // (past the run's last piece the loads still run, so that the waits count the same loads
        // every step, but against an empty buffer: zeros land and nothing is fetched; the same
        // for the rows a share of the last rows does not have)
        const uint32_t o = load_tile / PER;
        // (and for the pieces past the row that the last stretch of one that does not divide has)
        const bool beyond = LONG && !SPLIT && 1024u * NP * kpart + 128u * (NP * wave + load_piece) >= a.row_bytes;
        const __amdgpu_buffer_rsrc_t buf = o < count && !beyond ? wbuf : nobuf;
        const uint32_t base = (first_row(o) + (PAIR && (load_tile & 1u) ? a.half : 0u)) * a.row_bytes + 128u * load_piece, rows = rows_of(o);
        const uint32_t dst = ring0 + load_slot * (WAVES * SLOT);
#pragma unroll
        for (int j = 0; j < LOADS; j++) load_lds_b128(8u * j < rows ? buf : nobuf, dst + 1024u * j, woff[j] + base);
        load_piece = load_piece + 1u == (uint32_t)NP ? 0u : load_piece + 1u;
        load_tile += load_piece == 0u ? 1u : 0u;
        load_slot = (load_slot + 1u) % DEPTH;
    };

    // The tokens' inputs first: loads complete in order within a wave, and behind the weight
    // loads the first use of an input would wait for a round trip of the weight stream. Operand
    // row r of the matrix instruction is piece r / 8 of token 4 (r / 4 % 2) + r % 4 (rows 24 .. 31
    // are zeros), so that a lane's sixteen results are its weight row times the three pieces of
    // four tokens; the lane's eight positions of step s are 16 s + 8 (lane / 32) ... An absent
    // token's rows read the last token's inputs and come out as zeros: no branches, so all of the
    // lane's loads go out together.
    const uint32_t rho = lane & 31u, kap = lane >> 5;
    const uint32_t tok = 4u * ((rho >> 2) & 1u) + (rho & 3u), piece = rho >> 3;
    const bool live = tok < a.m && piece < PIECES;
    hu32x4 xf[4 * NP];
    if constexpr (SPLIT) {
        // Every step's operand is sixteen bytes of a plane; the lanes of absent tokens and of
        // the zero rows ask past the buffer's end and get zeros.
        const __amdgpu_buffer_rsrc_t pbuf = make_buffer(q.planes, PIECES * q.plane_tokens * q.plane_k * 2u);
        const uint32_t at = live ? ((piece * q.plane_tokens + q.t0 + tok) * q.plane_k + q.plane_first + 512u * NP * kpart + 64u * NP * wave + 8u * kap) * 2u : 0xfffffff0u;
#pragma unroll
        for (int s = 0; s < 4 * NP; s++) xf[s] = __builtin_bit_cast(hu32x4, __builtin_amdgcn_raw_buffer_load_b128(pbuf, live ? at + 32u * s : at, 0, 0));
        issue();
#pragma unroll
        for (int s = 1; s < DEPTH - 1; s++) issue();
    } else {
        // Wave w takes token w, lane l its vectors l, l + 64, ... (a wave without a token reads an
        // empty buffer). A token's values depend on nothing but its inputs.
        constexpr uint32_t ROW = piece_row<NP>(), PIECES_AT = (LDS_BYTES - 64u - pieces_bytes<NP, PIECES>()) & ~15u;
        constexpr uint32_t FREE = PIECES_AT < PART_BYTES ? 0u : (PIECES_AT - PART_BYTES) / (WAVES * SLOT);
        constexpr int EARLY = FREE < DEPTH - 1 ? FREE : DEPTH - 1;  // pieces of weights asked for meanwhile
        const __amdgpu_buffer_rsrc_t xbuf = make_buffer(a.x + (wave < a.m ? (size_t)wave * a.xr : 0u) + 512u * NP * kpart, wave < a.m ? 4u * min(a.k, a.row_bytes / 2u - 512u * NP * kpart) : 0u);
        const __amdgpu_buffer_rsrc_t gbuf = make_buffer(a.norm_w, (a.flags & FLAG_NORM) && wave < a.m ? 4u * a.k : 0u);
        float4 v[2 * NP], g[2 * NP];
#pragma unroll
        for (int j = 0; j < 2 * NP; j++) v[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, 16u * (lane + 64u * j), 0, 0));
        if (a.flags & FLAG_NORM) {
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) g[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(gbuf, 16u * (lane + 64u * j), 0, 0));
        }
#pragma unroll
        for (int s = 0; s < EARLY; s++) issue();
        if (a.flags & FLAG_NORM) {
            // (stage_token's additions: its wave w takes the vectors of every fourth j from w on, so that a
            // token is the same bits however it is staged; a single chain of all of them would be four times as long)
            float ss[4] = {};
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) ss[j & 3] += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
#pragma unroll
            for (int w = 0; w < 4; w++) ss[w] = wave_sum(ss[w]);
            const float scale = 1.0f / sqrtf(((ss[0] + ss[1]) + (ss[2] + ss[3])) / (float)a.k + a.eps);
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) {
                v[j].x = v[j].x * scale * g[j].x; v[j].y = v[j].y * scale * g[j].y;
                v[j].z = v[j].z * scale * g[j].z; v[j].w = v[j].w * scale * g[j].w;
            }
        }
        uint8_t *mine = lds + PIECES_AT + wave * ROW;
        if constexpr (F16) {
            float big = 0.f;
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) big = largest<false>(big, v[j]);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off, 64));
            if (big == __builtin_inff()) {
                big = 0.f;
#pragma unroll
                for (int j = 0; j < 2 * NP; j++) big = largest<true>(big, v[j]);
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off, 64));
            }
            float scale, inverse;
            f16_scale(big, scale, inverse);
            if (lane == 0) lds_inverse[wave] = inverse;
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) {
                uint2 w[PIECES];
                f16_pieces<PIECES>(v[j], scale, w);
#pragma unroll
                for (uint32_t p = 0; p < PIECES; p++) *reinterpret_cast<uint2 *>(mine + 8u * p * ROW + 8u * (lane + 64u * j)) = w[p];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 2 * NP; j++) {
#pragma unroll
                for (uint32_t p = 0; p < 3u; p++) *reinterpret_cast<uint2 *>(mine + 8u * p * ROW + 8u * (lane + 64u * j)) = bf16_piece(v[j], p);
            }
        }
        lds_barrier();
        const uint8_t *from = lds + PIECES_AT + ((live ? 8u * piece + tok : 0u) * ROW) + 2u * (64u * NP * wave + 8u * kap);
#pragma unroll
        for (int s = 0; s < 4 * NP; s++) {
            const hu32x4 w = *reinterpret_cast<const hu32x4 *>(from + 32u * s);
#pragma unroll
            for (int e = 0; e < 4; e++) xf[s][e] = live ? w[e] : 0u;
        }
        lds_barrier();  // (the ring, the partial sums and the kept outputs lie where the pieces were)
#pragma unroll
        for (int s = EARLY; s < DEPTH - 1; s++) issue();
    }

    // The lane's reads of a piece: row rho, chunk 2 s + kap of its line for step s.
    uint32_t r_at[4];
#pragma unroll
    for (int s = 0; s < 4; s++) r_at[s] = 128u * rho + 16u * ((2u * s + kap) ^ line_key(rho));

    auto finish = [&](uint32_t p, const hf32x16 &sum) __attribute__((always_inline)) {
        float *part = lds_part + (p & 1u) * (WAVES * 256u);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float all = !F16 ? (sum[i] + sum[4 + i]) + sum[8 + i] : fmaf(PIECES == 3 ? fmaf(sum[8 + i], 1.0f / 2048.0f, sum[4 + i]) : sum[4 + i], 1.0f / 2048.0f, sum[i]);
            // (an infinite weight makes an infinity of an input's first piece, but NaNs of pieces that are zero)
            part[wave * 256u + 64u * i + lane] = fabsf(sum[i]) == __builtin_inff() ? sum[i] : all;
        }
        lds_barrier();
        // Buffer p % 2 is written again in step p + 2, after the barrier of step p + 1, which a
        // wave passes only when it has read what it needs here. The 256 outputs of a tile are
        // summed by one half of the workgroup, the other half at the next tile.
        if ((tid >> 8) == (p & 1u)) {
            // (a wave sums tokens i and 4 + i, whose partial sums lie side by side: no two lanes on a bank)
            const uint32_t row = tid & 31u, tk = 4u * ((tid >> 5) & 1u) + ((tid >> 6) & 3u);
            const float *src = part + 64u * (tk & 3u) + 32u * (tk >> 2) + row;
            static_assert(WAVES == 8, "the sum below");
            float total = ((src[0] + src[256u]) + (src[512u] + src[768u])) + ((src[1024u] + src[1280u]) + (src[1536u] + src[1792u]));
            if (F16) total *= lds_inverse[tk];
            // (PAIR: the gate tile's output waits here for the up tile's, a barrier later)
            float *kept = lds_kept + 256u * (p / PER % KEPT) + 32u * tk + row;
            *kept = PAIR && (p & 1u) ? silu_f(*kept) * total : total;
        }
    };
    // The outputs of output tiles first .. first + n - 1, from LDS to memory: 128 contiguous bytes a
    // token and tile. (Stored tile by tile between the loads they took 2 us of a 55 us launch
    // longer than in one burst: every isolated write turns the memory's direction around.)
    auto store_kept = [&](uint32_t first, uint32_t n) __attribute__((always_inline)) {
        lds_barrier();
        for (uint32_t p = first + (tid >> 8); p < first + n; p += 2u) {
            const uint32_t row = tid & 31u, tk = (tid >> 5) & 7u;
            const uint32_t j = first_row(p) + row;
            if (tk < a.m && row < rows_of(p) && j < a.rows) {
                float *o = a.out + (size_t)tk * a.out_stride + a.col0 + j;
                const float total = lds_kept[256u * (p % KEPT) + (tid & 255u)];
                if (LONG) store_apart(q.partial + ((size_t)kpart * 8u + tk) * a.rows + j, total);
                else store_apart(o, (a.flags & FLAG_ACCUMULATE) ? *o + total : total);
            }
        }
    };

    // DEPTH ring slots in rotation. Every wave of the workgroup runs the same steps (the barrier
    // inside). Before a piece is read, all but the loads of the DEPTH - 1 pieces after it have
    // landed.
    uint32_t slot = 0;
    for (uint32_t p = 0; p < PER * count; p++) {
        hf32x16 sum;
#pragma unroll
        for (int e = 0; e < 16; e++) sum[e] = 0.f;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            // The slot refilled now was read by the multiply before: its reads must have returned
            // before the load is issued (a load past the run's end lands at once), and the
            // compiler, which sees no dependency between the two, must not move it up.
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue();
            wait_loads<(DEPTH - 1) * LOADS>();
            const uint8_t *t = ring + slot * (WAVES * SLOT);
            hf32x16 part;
#pragma unroll
            for (int e = 0; e < 16; e++) part[e] = 0.f;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const hu32x4 w = *reinterpret_cast<const hu32x4 *>(t + r_at[s]);
                if constexpr (F16) part = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(hf16x8, xf[4 * i + s]), __builtin_bit_cast(hf16x8, w), part, 0, 0, 0);
                else part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(hbf16x8, xf[4 * i + s]), __builtin_bit_cast(hbf16x8, w), part, 0, 0, 0);
            }
            // (the piece's matrix instructions belong here, not after the last piece's wait, where
            // the compiler would otherwise collect them with all their operands held in registers)
            asm volatile("" : "+v"(part));
#pragma unroll
            for (int e = 0; e < 4 * (int)PIECES; e++) sum[e] = i == 0 ? part[e] : sum[e] + part[e];
            slot = (slot + 1u) % DEPTH;
        }
        finish(p, sum);
        // (the next tile's sums are kept only behind its barrier, which no thread passes before
        // it has stored what it stores here)
        const uint32_t o = p / PER;
        if ((!PAIR || (p & 1u)) && ((o + 1u) % KEPT == 0u || o + 1u == count)) store_kept(o - o % KEPT, o % KEPT + 1u);
    }
    wait_loads<0>();  // nothing may still land in LDS once the workgroup is gone
}

// Token blockIdx.x as the multiply sees it (normalised if the step asks for it:
// src/kernels/matvec_half.wgsl:58-80), split into the three planes.
__global__ __launch_bounds__(256) void matvec_bf16_split_kernel(MvArgs a, uint2 *planes) {
    __shared__ float red[4];
    extern __shared__ float4 staged[];  // the token: k / 4 vectors
    stage_token(a, blockIdx.x, staged, red);
    __syncthreads();
    const uint32_t k4 = a.k / 4u;
    for (uint32_t i = threadIdx.x; i < k4; i += 256u) {
        const float4 v = staged[i];
#pragma unroll
        for (uint32_t piece = 0; piece < 3u; piece++) planes[(size_t)(piece * gridDim.x + blockIdx.x) * k4 + i] = bf16_piece(v, piece);
    }
}

// The same for matvec_f16: the token scaled by the power of two that puts its largest
// magnitude in [2^14, 2^15) and split into PIECES f16 values a weight (planes
// [piece][tokens][k]), and one over the scale.
template <uint32_t PIECES>
__global__ __launch_bounds__(256) void matvec_f16_split_kernel(MvArgs a, uint2 *planes, float *inverse) {
    __shared__ float red[4];
    extern __shared__ float4 staged[];  // the token: k / 4 vectors
    stage_token(a, blockIdx.x, staged, red);
    __syncthreads();
    const uint32_t tid = threadIdx.x, k4 = a.k / 4u;
    float big = 0.f;
    for (uint32_t i = tid; i < k4; i += 256u) big = largest<true>(big, staged[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off, 64));
    if ((tid & 63u) == 0) red[tid >> 6] = big;
    __syncthreads();
    big = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float scale, inv;
    f16_scale(big, scale, inv);
    if (tid == 0) inverse[blockIdx.x] = inv;
    for (uint32_t i = tid; i < k4; i += 256u) {
        uint2 w[PIECES];
        f16_pieces<PIECES>(staged[i], scale, w);
#pragma unroll
        for (uint32_t p = 0; p < PIECES; p++) planes[(size_t)(p * gridDim.x + blockIdx.x) * k4 + i] = w[p];
    }
}

template <int NP, bool SPLIT, bool F16, bool LONG, bool PAIR, bool WHOLE>
zhip_result launch_blocks(const Dispatch &d, const StreamArgs &q, dim3 grid) {
    auto kernel = matvec_bf16_mfma_stream_kernel<NP, SPLIT, F16, LONG, PAIR, WHOLE>;
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) != hipSuccess) {
            (void)hipGetLastError();
            return fail(d, ZHIP_E_GPU, "%s: cannot reserve %u bytes of LDS", F16 ? "matvec_f16" : "matvec_bf16", LDS_BYTES);
        }
        configured = true;
    }
    const uint32_t walkers = grid.x / q.parts;
    if (!MV_HOLDS(q.a) || (q.rounds | walkers | q.tail_rem) > 0xffffu || (q.tail_base | q.a.m) > 15u || q.parts > 127u) return fail(d, ZHIP_E_GPU, "%s: %u rounds of %u workgroups", F16 ? "matvec_f16" : "matvec_bf16", q.rounds, walkers);
    hipLaunchKernelGGL(kernel, grid, dim3(THREADS), LDS_BYTES, d.stream, q.a.x, q.a.w, q.a.norm_w, q.a.k | q.a.flags << 24, q.a.xr, q.a.row_bytes, q.a.rows, q.a.half, q.w_bytes,
        q.rounds | walkers << 16, q.tail_rem | q.tail_base << 16 | q.a.m << 20 | q.by_die << 24 | q.parts << 25, q);
    return check_launch(d, F16 ? "matvec_f16" : "matvec_bf16");
}

}  // namespace

// Whether this kernel can run the (already validated) arguments: k split into whole lines a
// wave, and rows of whole lines where the workgroups split the tokens of long ones themselves (`own` below); a gate / up pair only over rows that one workgroup takes whole.
// (rows of more than 4096 weights are taken in stretches of columns: equal ones in one launch, workgroups sharing a
// tile, with a launch for their sums; unequal ones behind the RMSNorm prologue a launch each; up to 16384: the split launch stages a token in 64 KB of LDS)
// (32-bit byte offsets up to a tile past the last row: larger matrices are the general kernel's)
bool matvec_bf16_mfma_stream_accepts(const MvArgs &a) {
    const bool pair = a.flags & FLAG_SILU_PAIR;
    if ((pair && a.k > 4096u) || ((pair ? (uint64_t)a.half : 0ull) + a.rows + 64u) * a.row_bytes >= 0xfffffff0ull) return false;
    return a.m >= 1 && a.k >= 1024u && a.k <= 16384u && (a.k % 512u == 0 || (a.k % 64u == 0 && a.k > 4096u && !(a.flags & FLAG_NORM))) && a.act_div == 0.f && a.rows >= 1 &&
           a.xr % 4u == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15u) == 0 && a.row_bytes == 2u * a.k;
}

// The stretches' lengths, in 512 columns: rows of up to 4096 weights 2 .. 8, longer rows 4 .. 8 behind the RMSNorm prologue (equal ones 5 .. 8), 3 .. 6 without.
template <int NP, bool SPLIT, bool F16, bool LONG, bool PAIR, bool WHOLE>
static zhip_result launch_np(const Dispatch &d, const StreamArgs &q, dim3 grid) {
    constexpr int LOW = LONG ? (SPLIT ? 5 : 3) : SPLIT ? 4 : 2, HIGH = LONG && !SPLIT ? 6 : 8;
    if constexpr (NP >= LOW && NP <= HIGH) {
        if (q.a.k == 512u * NP) return launch_blocks<NP, SPLIT || !pieces_fit<NP, pieces_of(F16, WHOLE)>(), F16, LONG, PAIR, WHOLE>(d, q, grid);
    }
    if constexpr (NP < 8) return launch_np<NP + 1, SPLIT, F16, LONG, PAIR, WHOLE>(d, q, grid);
    else return fail(d, ZHIP_E_GPU, "%s: a stretch of %u columns", F16 ? "matvec_f16" : "matvec_bf16", q.a.k);
}
template <bool SPLIT, bool F16, bool LONG = false, bool PAIR = false, bool WHOLE = PAIR>
static zhip_result launch_for_k(const Dispatch &d, const StreamArgs &q, dim3 grid) { return launch_np<2, SPLIT, F16, LONG, PAIR, WHOLE>(d, q, grid); }

// f16: the weights are f16 (matvec_f16), bf16 otherwise.
zhip_result launch_matvec_bf16_mfma_stream(const Dispatch &d, const MvArgs &a, uint64_t w_bytes, bool f16) {
    const char *name = f16 ? "matvec_f16" : "matvec_bf16";
    const bool pair = a.flags & FLAG_SILU_PAIR;
    const uint64_t used = ((uint64_t)a.rows + (pair ? a.half : 0u)) * a.row_bytes;
    const uint32_t cus = (uint32_t)d.dev->compute_units;
    const uint32_t units = (a.rows + 7u) / 8u;
    const uint32_t groups = units < cus ? units : cus;
    const uint32_t rounds = (a.rows / 32u) / groups;
    const uint32_t tail = (a.rows - 32u * rounds * groups + 7u) / 8u;
    StreamArgs q{a, (uint32_t)(used < w_bytes ? used : w_bytes), rounds, tail / groups, tail % groups, groups % 8u == 0 ? 1u : 0u, nullptr, 0u, 0u, 0u, 0u, nullptr, 1u, nullptr};
    // Rows of more than 4096 weights (the FFN-down shapes; the general kernel takes them token by
    // token) go in stretches of columns, by two rules: behind the RMSNorm prologue as few of up to 4096 as there can be (14336 = 4 x 3584, 8192 =
    // 2 x 4096, 9728 = 3584 + 2 x 3072), without it see below (7 x 2048, 4 x 2048, 4 x 2560 less 512). Together in
    // one launch, `launches` workgroups share a walker's tiles, a
    // stretch each, and a second launch adds the stretches' sums in their order and applies the
    // epilogue (their sums wait in the workspace, behind the tokens' planes where there are any).
    const uint32_t token_pieces = pieces_of(f16, pair), pieces = (a.k + 511u) / 512u, fits = token_pieces == 2u ? 8u : 6u;
    uint32_t launches = (a.k + 4095u) / 4096u;
    // Without the RMSNorm prologue the workgroups split their stretches' tokens themselves: in stretches of up to 3072 columns
    // (what fits LDS in bf16, and in f16 the sums are the shorter ones), equal ones where two more than the fewest at most are, or with a last one that ends past the
    // row. Behind the prologue the tokens are split (and normalised) by a launch of their own, and so are those of
    // shorter rows whose pieces do not fit (three of them a token above 3072 weights). us at one / four / eight tokens, ACCUMULATE,
    // split in front / by the workgroups:
    //   2048 x 8192 f16    18.4 19.2 20.2 / 13.1 13.3 13.2    bf16 17.6 19.1 21.2 / 13.0 13.2 13.0
    //   2560 x 9728        31.8 33.1 35.6 / 16.3 16.4 16.5         30.5 32.6 38.7 / 17.2 17.7 18.0   (unequal: a launch a stretch)
    //   4096 x 14336       32.7 33.4 34.2 / 27.7 27.7 27.5         31.9 32.9 34.5 / 27.6 27.5 27.5
    //   2048 x 5120        14.0 14.7 15.6 / 11.2 11.3 11.3         13.4 14.6 16.6 / 11.5 11.6 11.7
    // (f16 in two stretches of 4096, 2048 x 8192: 14.6 15.0 15.1; in three of 3584, 2560 x 9728: 16.6 16.8 17.0; relative
    // errors as before, 1.02e-7 .. 1.11e-7, bf16 8.7e-8 .. 9.7e-8)
    const uint32_t fewest = (pieces + 5u) / 6u;
    const bool own = launches > 1u && !(a.flags & FLAG_NORM) && fewest + 2u <= kMatvecMaxParts && fewest + 2u <= cus;
    if (own) {
        launches = fewest;
        for (uint32_t n = fewest + 2u; n >= fewest; n--) launches = pieces % n == 0u ? n : launches;
    }
    // (an input keeps all its bits where the general kernel was the alternative)
    const bool whole = a.k % 512u != 0 || (uint64_t)a.rows * a.row_bytes < kMatvecBf16StreamBytes;
    const bool split = !own && pieces > fits;
    const bool together = own || (launches > 1u && pieces % launches == 0u && split && launches <= kMatvecMaxParts && cus >= launches);
    const uint64_t planes_bytes = own ? 0ull : ((2ull * token_pieces * a.m * a.k + 4ull * a.m + 64u) + 255u) & ~255ull;
    if (own) {
        if (!d.work) return fail(d, ZHIP_E_GPU, "%s: no workspace", name);
        if (zhip_result r = d.work->reserve(d, (uint64_t)launches * 8u * a.rows * sizeof(float))) return r;
    }
    if (split) {
        const uint64_t bytes = 2ull * token_pieces * a.m * a.k;
        if (!d.work) return fail(d, ZHIP_E_GPU, "%s: no workspace", name);
        if (bytes >= 0xfffffff0ull) return fail(d, ZHIP_E_BAD_COMMAND, "%s: a step of %u tokens", name, a.m);
        if (zhip_result r = d.work->reserve(d, planes_bytes + (together ? (uint64_t)launches * 8u * a.rows * sizeof(float) : 0ull))) return r;
        float *inverse = reinterpret_cast<float *>(d.work->data + bytes);
        if (f16 && pair) hipLaunchKernelGGL(matvec_f16_split_kernel<3>, dim3(a.m), dim3(256), a.k * 4u, d.stream, a, reinterpret_cast<uint2 *>(d.work->data), inverse);
        else if (f16) hipLaunchKernelGGL(matvec_f16_split_kernel<2>, dim3(a.m), dim3(256), a.k * 4u, d.stream, a, reinterpret_cast<uint2 *>(d.work->data), inverse);
        else hipLaunchKernelGGL(matvec_bf16_split_kernel, dim3(a.m), dim3(256), a.k * 4u, d.stream, a, reinterpret_cast<uint2 *>(d.work->data));
        if (zhip_result r = check_launch(d, name)) return r;
        q.planes = d.work->data;
        q.plane_tokens = a.m;
        q.plane_k = a.k;
        q.inverse = inverse;
        q.a.flags &= ~FLAG_NORM;
        q.a.norm_w = nullptr;
    }
    const dim3 grid(groups);
    // Stretches of unequal length: each a launch that adds to the one before; the tokens are
    // split once, prologue included, for all of them.
    if (together) {
        const uint32_t most = cus / launches, walkers = units < most ? units : most;
        const uint32_t lrounds = (a.rows / 32u) / walkers, ltail = (a.rows - 32u * lrounds * walkers + 7u) / 8u;
        q.rounds = lrounds; q.tail_base = ltail / walkers; q.tail_rem = ltail % walkers; q.by_die = walkers % 8u == 0 ? 1u : 0u;
        q.parts = launches;
        q.partial = reinterpret_cast<float *>(d.work->data + planes_bytes);
        q.a.k = 512u * ((pieces + launches - 1u) / launches);
        q.plane_first = 0;
        for (uint32_t t0 = 0; t0 < a.m; t0 += 8u) {
            q.a.x = a.x + (size_t)t0 * a.xr;
            q.a.out = a.out + (size_t)t0 * a.out_stride;
            q.a.m = a.m - t0 < 8u ? a.m - t0 : 8u;
            q.a.flags = a.flags & ~FLAG_NORM;
            q.t0 = t0;
            const dim3 all(walkers * launches);
            zhip_result r;
            if (own && f16) r = whole ? launch_for_k<false, true, true, false, true>(d, q, all) : launch_for_k<false, true, true>(d, q, all);
            else if (own) r = launch_for_k<false, false, true>(d, q, all);
            else r = f16 ? launch_for_k<true, true, true>(d, q, all) : launch_for_k<true, false, true>(d, q, all);
            if (r != ZHIP_OK) return r;
            MvArgs sum = q.a;
            sum.k = a.k;
            if ((r = launch_matvec_parts_sum(d, name, sum, q.partial, launches)) != ZHIP_OK) return r;
        }
        return ZHIP_OK;
    }
    for (uint32_t t0 = 0; t0 < a.m; t0 += 8u) {
        uint32_t first = 0;
        for (uint32_t c = 0; c < launches; c++) {
            q.a.k = 512u * (pieces / launches + (c < pieces % launches ? 1u : 0u));
            q.a.x = a.x + (size_t)t0 * a.xr + first;
            q.a.w = a.w + 2u * (size_t)first;
            q.w_bytes = (uint32_t)((used < w_bytes ? used : w_bytes) - 2u * (uint64_t)first);
            q.a.out = a.out + (size_t)t0 * a.out_stride;
            q.a.m = a.m - t0 < 8u ? a.m - t0 : 8u;
            q.a.flags = (a.flags & ~FLAG_NORM & ~FLAG_ACCUMULATE) | ((c || (a.flags & FLAG_ACCUMULATE)) ? FLAG_ACCUMULATE : 0u);
            if (!split) {
                q.a.flags = a.flags;
                q.a.norm_w = a.norm_w;
            }
            q.t0 = t0;
            q.plane_first = first;
            zhip_result r;
            if (pair) {
                if (f16) r = launch_for_k<false, true, false, true>(d, q, grid);
                else r = launch_for_k<false, false, false, true>(d, q, grid);  // (above 3072 weights that is the split tokens' kernel)
            } else if (f16) r = split ? launch_for_k<true, true>(d, q, grid) : launch_for_k<false, true>(d, q, grid);
            else r = split ? launch_for_k<true, false>(d, q, grid) : launch_for_k<false, false>(d, q, grid);
            if (r != ZHIP_OK) return r;
            first += q.a.k;
        }
    }
    return ZHIP_OK;
}

}  // namespace zhip
