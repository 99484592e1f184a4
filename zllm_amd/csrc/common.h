// Internal interface between the command-stream host and the gfx950 kernels.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/zllm_hip.h"

namespace zhip {

// Parameter blocks, field for field as src/kernels/kernels.zig:432-505 declares
// them (extern structs, little-endian, bound at binding 0).
struct MatvecParams {  // params.MatvecBf16
    uint32_t n, k, col0, out_stride;
    float eps;
    uint32_t flags;
    uint32_t half;
    uint32_t x_stride;  // vec4 units between tokens' inputs; 0: k / 4
};
enum : uint32_t { FLAG_NORM = 1u, FLAG_ACCUMULATE = 2u, FLAG_SILU_PAIR = 4u };

struct MatmulParams {  // params.MatmulBf16 / params.MatmulQuant
    uint32_t rows, n, k, col0, out_stride, accumulate;
    uint32_t k_slice;       // MatmulBf16: padding
    uint32_t slice_stride;  // MatmulBf16: padding
};

struct MatmulReduceParams {
    uint32_t rows, n, slices, col0, out_stride, accumulate, slice_stride, pad;
};

struct SiluMulParams { uint32_t count, width, pad0, pad1; };
struct RepackQ80Params { uint32_t rows, k, pad0, pad1; };
struct RepadParams { uint32_t blocks, src_bytes, dst_bytes, pad; };

static_assert(sizeof(MatvecParams) == 32, "params.MatvecBf16 is 32 bytes");
static_assert(sizeof(MatmulParams) == 32, "params.MatmulQuant is 32 bytes");
static_assert(sizeof(MatmulReduceParams) == 32, "params.MatmulReduce is 32 bytes");
static_assert(sizeof(SiluMulParams) == 16 && sizeof(RepackQ80Params) == 16 && sizeof(RepadParams) == 16, "16-byte blocks");

// A quantized decode multiply's tunables (kernels.MatvecVariant,
// src/kernels/kernels.zig:319-338), decoded from the create_kernel variant id.
struct MatvecVariant {
    uint32_t wg = 256, lanes = 32, rows = 1, act_div = 0;
    uint32_t groupRows() const { return wg / lanes * rows; }
};

// Steps of up to this many tokens may use the decode multiplies. The reference
// caps its kernels at 4 (src/kernels/matvec_quant.wgsl.hbs:64-65); rows 5..8
// are this backend's extension for speculative-verify widths.
constexpr uint32_t kMaxDecodeRows = 8;

// A byte offset no binding reaches (a binding is at most 2 GiB): a range-checked buffer load
// there returns zeros and moves nothing.
constexpr uint32_t kNowhere = 0xF0000000u;

// The longest step the reference's planner records (src/plan/plan.zig:129,
// src/plan/qwen35.zig:335).
constexpr uint32_t kPlannerStepCap = 512;

struct Bind {
    uint8_t *ptr = nullptr;  // buffer base + binding offset
    uint64_t size = 0;       // bytes bound
    bool bound = false;
};

struct DeviceInfo {
    int compute_units = 256;
    int max_lds = 65536;
    bool wide_decode = false;  // ZHIP_OPTION_WIDE_DECODE
};

struct Dispatch;

// Device scratch a launcher may ask for (the bf16 copy of a step's f32
// activations). Owned by the context, grown on demand, freed with the context.
// Everything runs on the context's one in-order stream, so consecutive
// dispatches can share it.
struct Workspace {
    uint8_t *data = nullptr;
    uint64_t bytes = 0;
    bool fixed = false;  // memory the workspace does not own: never grown, never freed
    bool used = false;   // asked for since this was last cleared
    bool kept = false;   // as it is: growing waits for the stream, which would end the capture of a graph
    Workspace *spare = nullptr;  // kSpareWorkspaces that are given up where memory is short of what this one needs
    uint64_t refused = ~0ull;  // reserve_quietly: the least that has not been there since this was last cleared
    // Makes at least `want` bytes available (fails on a fixed workspace that is too small).
    zhip_result reserve(const Dispatch &d, uint64_t want);
    // The same for what a launch can do without: null, and no message, if memory is short. Asked for once, not by every launch of a
    // step: growing waits for the launches before it.
    uint8_t *reserve_quietly(const Dispatch &d, uint64_t want);
    void release();
};
// The places of packed activations: two, one is read while the next is written. Nobody needs them where memory is short: a dispatch that asks for
// the workspace reads from neither, and between submits nothing is in them.
constexpr int kSpareWorkspaces = 2;
// hipMalloc, with what `spare` (kSpareWorkspaces of them, or null) hold where memory is short.
hipError_t allocate(void **p, uint64_t size, hipStream_t stream, Workspace *spare);

// Activations as a float rung's multiplies read them: two bytes a value, or two such planes (the rounded values and what each
// rounding left). Such a multiply packs its f32 activations in a pass of its own, unless the dispatch right before it
// wrote exactly those values: it has them in registers and stores them packed as well, the same roundings. A pass reads six bytes
// a value from L2 and is a launch that the multiply waits for. us a step, passes / packed by the writers: six layers of 4096 x
// 14336 with Q8_0 in bf16, 512 tokens, 2277 / 2187; twelve of 2048 x 6144 in f16, 128 tokens, 856 / 744; twelve of 1024 x 3072
// in bf16, 17 tokens, 420 / 330; in two f16 planes, 100 tokens, 933 / 874.
struct PackedCopy {
    enum Kind : uint32_t { none, bf16, f16, f16_split };
    static constexpr uint64_t kMost = 64u << 20;  // a writer packs up to here: 512 tokens of 65,536 values, in two planes 32,768
    const float *x = nullptr;  // rows x k values, dense
    uint32_t rows = 0, k = 0;
    Kind kind = none;
    Workspace *room = nullptr;
    uint8_t *data = nullptr;   // set once they have been written
    uint64_t plane() const { return ((uint64_t)rows * k * 2u + 255u) & ~255ull; }
    bool of(const float *p, uint32_t r, uint32_t c, Kind as) const { return kind == as && as != none && x == p && rows == r && k == c; }
    // Where their writer puts them: null if they are too many or memory is short (the multiply then packs them itself).
    uint8_t *reserve(const Dispatch &d) const;
};

// Activations as an int8 Q8_0 multiply reads them, rounded to 8-bit blocks of 32 by a quantize_q8 dispatch. Where such a multiply
// writes them, that dispatch is the next and another such multiply the one behind it, the first rounds what it stores, into a
// place aside (it may still be reading the last rounding where the next one belongs), the quantize_q8 launch is left out, and the
// second multiplies from there and puts the rounding where the caller has it. Two launches fewer a layer, and a SiLU pair's values are not
// read back. See matmul_q8_i8.hip for what it measured.
struct RoundedCopy {
    static constexpr uint64_t kMost = 64u << 20;  // 512 tokens of 116,000 values
    const float *x = nullptr;  // rows x k values, dense (mode 2: rows x 2 k)
    uint32_t rows = 0, k = 0, mode = 0;
    uint8_t *q = nullptr, *d = nullptr;  // the caller's values and scales
    Workspace *room = nullptr;
    uint8_t *data = nullptr;  // set once they have been rounded: the values, and scales_at() behind them the scales
    uint64_t scales_at() const { return ((uint64_t)rows * k + 255u) & ~255ull; }
    uint64_t scales_bytes() const { return (uint64_t)rows * (k / 32u) * 4u; }
    uint8_t *reserve(const Dispatch &d) const;
};
// What an int8 Q8_0 multiply's launch touches, where it is one that can read them so.
struct RoundedRead {
    const uint8_t *q = nullptr, *d = nullptr, *w = nullptr, *out = nullptr;
    uint32_t rows = 0, k = 0;
    uint64_t w_bytes = 0, out_bytes = 0;
};

// One resolved dispatch: binding 0's bytes come from the host's shadow copy of
// the uniform buffer, so kernels take their parameters by value.
struct Dispatch {
    const uint8_t *params = nullptr;
    size_t params_size = 0;
    Bind bind[8];
    uint32_t grid[3] = {0, 0, 0};
    uint32_t variant = 0;
    hipStream_t stream = nullptr;
    const DeviceInfo *dev = nullptr;
    Workspace *work = nullptr;
    PackedCopy *wanted = nullptr;      // a float rung's multiply: nothing is launched, what it would pack is left there
    PackedCopy *next = nullptr;        // what the dispatch behind this one would pack
    const PackedCopy *have = nullptr;  // what the dispatch before this one has packed
    RoundedCopy *rounds = nullptr;         // quantize_q8: nothing is launched, what it would round is left there
    RoundedRead *reads = nullptr;          // matmul_q8_0: the same
    RoundedCopy *rounded_out = nullptr;    // what the quantize_q8 behind this dispatch would round
    const RoundedCopy *rounded_in = nullptr;  // what the multiply before the last dispatch has rounded
    char *err = nullptr;  // message buffer for a failed launch
    size_t err_cap = 0;
};

// Launches one kernel for a dispatch, after checking that the bound ranges
// cover everything the kernel will touch. Returns ZHIP_OK, ZHIP_E_BAD_COMMAND
// (with a message) or ZHIP_E_GPU.
typedef zhip_result (*LaunchFn)(const Dispatch &);

zhip_result launch_matvec_q8_0(const Dispatch &);
zhip_result launch_matvec_q3_k(const Dispatch &);
zhip_result launch_matvec_q4_k(const Dispatch &);
zhip_result launch_matvec_q5_k(const Dispatch &);
zhip_result launch_matvec_q6_k(const Dispatch &);
zhip_result launch_matvec_bf16(const Dispatch &);
zhip_result launch_matvec_f16(const Dispatch &);
zhip_result launch_matmul_reduce(const Dispatch &);
zhip_result launch_quantize_q8(const Dispatch &);
zhip_result launch_matmul_q8_0(const Dispatch &);
zhip_result launch_matmul_q3_k(const Dispatch &);
zhip_result launch_matmul_q4_k(const Dispatch &);
zhip_result launch_matmul_q5_k(const Dispatch &);
zhip_result launch_matmul_q6_k(const Dispatch &);
zhip_result launch_silu_mul(const Dispatch &);
zhip_result launch_repack_q8_0(const Dispatch &);
zhip_result launch_repack_q3_k(const Dispatch &);
zhip_result launch_repad(const Dispatch &);
zhip_result launch_embed_q8_0(const Dispatch &);
zhip_result launch_embed_q3_k(const Dispatch &);
zhip_result launch_embed_q4_k(const Dispatch &);
zhip_result launch_embed_q5_k(const Dispatch &);
zhip_result launch_embed_q6_k(const Dispatch &);
zhip_result launch_embed_bf16(const Dispatch &);
zhip_result launch_embed_f16(const Dispatch &);
zhip_result launch_embed_iq4_xs(const Dispatch &);

// Dynamic LDS above 64 KiB needs opting in once per kernel: done the first time this is called
// for the kernel (or ahead of time, see prepare_no_alloc_kernels), remembered after.
template <auto Kernel, int Bytes>
inline bool lds_opt_in() {
    static const bool ok = [] {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Bytes) == hipSuccess) return true;
        (void)hipGetLastError();
        return false;
    }();
    return ok;
}

// Host-side helpers shared by the launchers.
zhip_result fail(const Dispatch &d, zhip_result code, const char *fmt, ...);
zhip_result check_launch(const Dispatch &d, const char *kernel);

// The entry point that allocates nothing (no_alloc.hip): its fixed scratch array's address is
// looked up once per device, with that device current.
zhip_result no_alloc_setup(int device, const DeviceInfo &info);
// The one-time set-up of every kernel that entry point can launch (each file its own), so
// that the call itself does none.
bool matmul_mfma_prepare_no_alloc();
bool matmul_mfma_wide_prepare_no_alloc();
bool matmul_stream_prepare_no_alloc();
bool matmul_q8_bf16_prepare_no_alloc();
bool matmul_q8_bf16_wide_prepare_no_alloc();
uint64_t no_alloc_capacity();
zhip_result no_alloc_matmul_q8_0_float(int device, hipStream_t stream, const float *x, const void *w, float *out, uint32_t rows, uint32_t n,
    uint32_t k, uint32_t col0, uint32_t out_stride, uint32_t accumulate, char *err, size_t err_cap);

// Fills `words` 32-bit words at dst with `value` on the stream (clear_buffer;
// also used instead of memset nodes so a captured stream stays replayable).
zhip_result launch_fill(hipStream_t stream, void *dst, uint64_t words, uint32_t value);
// Copies `bytes` (a multiple of 4; both ends 4-byte aligned) between device and pinned host memory.
// (`stamp`, pinned or null, receives the GPU's clock; 0 bytes: that alone)
zhip_result launch_copy(hipStream_t stream, void *dst, const void *src, uint64_t bytes, uint64_t *stamp);
// Reads `bytes` to pinned memory in pieces: read_kernel, elementwise.hip.
zhip_result launch_read(hipStream_t stream, void *dst, const void *src, uint64_t bytes, uint64_t piece, uint32_t *arrived, uint64_t *flags, uint64_t ticket, uint64_t *first, uint64_t *last);

// A launch's time by its workgroups, where two share a CU: a lone one's time, and a pair's, which is less than twice
// that. An odd one out costs its CU a lone one's.
struct SharedCu {
    uint32_t lone, pair;
    constexpr uint64_t of(uint64_t workgroups, uint64_t cus) const {
        const uint64_t w = (workgroups + cus - 1u) / cus;
        return lone * (w & 1u) + pair * (w >> 1);
    }
};

}  // namespace zhip
