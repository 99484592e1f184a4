// Device scratch of a context: what its launchers' kernels leave for one another (common.h).
#include "common.h"

namespace zhip {

hipError_t allocate(void **p, uint64_t size, hipStream_t stream, Workspace *spare) {
    hipError_t e = hipMalloc(p, size);
    for (int i = 0; spare && i < kSpareWorkspaces && e == hipErrorOutOfMemory; i++) {
        if (!spare[i].data || hipStreamSynchronize(stream) != hipSuccess) continue;
        (void)hipGetLastError();
        spare[i].release();
        e = hipMalloc(p, size);
    }
    return e;
}

// Growing replaces the allocation, so earlier dispatches that may still be
// running with the old one are waited for first.
zhip_result Workspace::reserve(const Dispatch &d, uint64_t want) {
    used = true;
    if (want <= bytes) return ZHIP_OK;
    if (fixed) return fail(d, ZHIP_E_BAD_COMMAND, "workspace: %llu bytes wanted, the fixed scratch holds %llu", (unsigned long long)want, (unsigned long long)bytes);
    if (kept) return fail(d, ZHIP_E_GPU, "workspace: %llu bytes wanted during a capture, there are %llu", (unsigned long long)want, (unsigned long long)bytes);
    const uint64_t size = (want + (8u << 20) - 1) & ~(uint64_t)((8u << 20) - 1);
    if (hipStreamSynchronize(d.stream) != hipSuccess) return fail(d, ZHIP_E_GPU, "workspace: stream synchronisation failed");
    if (data) (void)hipFree(data);
    data = nullptr;
    bytes = 0;
    const hipError_t e = allocate(reinterpret_cast<void **>(&data), size, d.stream, spare);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        data = nullptr;
        return fail(d, e == hipErrorOutOfMemory ? ZHIP_E_OUT_OF_MEMORY : ZHIP_E_GPU, "workspace: cannot allocate %llu bytes", (unsigned long long)size);
    }
    bytes = size;
    return ZHIP_OK;
}

uint8_t *Workspace::reserve_quietly(const Dispatch &d, uint64_t want) {
    if (want >= refused) return nullptr;
    Dispatch quiet = d;
    quiet.err_cap = 0;
    if (reserve(quiet, want) == ZHIP_OK) return data;
    if (!kept) refused = want;
    return nullptr;
}

void Workspace::release() {
    if (data && !fixed) (void)hipFree(data);
    data = nullptr;
    bytes = 0;
}

uint8_t *PackedCopy::reserve(const Dispatch &d) const {
    const uint64_t want = kind == f16_split ? 2u * plane() : plane();
    return room && want <= kMost ? room->reserve_quietly(d, want) : nullptr;
}

uint8_t *RoundedCopy::reserve(const Dispatch &d) const {
    const uint64_t want = scales_at() + scales_bytes();
    return room && want <= kMost ? room->reserve_quietly(d, want) : nullptr;
}

}  // namespace zhip
