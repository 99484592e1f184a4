"""A context's device scratch (zllm_amd/csrc/workspace.cpp) on the CPU, built with g++ against a HIP of its own: what
growing calls, what a capture or a shortage of memory leaves out."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zllm_amd", "csrc")

PROGRAM = r"""
#include "common.h"
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <string>
using namespace zhip;

static std::string calls;  // s: synchronised, m: allocated, x: refused, f: freed
static uint64_t most = ~0ull;
static std::function<uint64_t()> held_by;
static uintptr_t next_address = 1u << 20;
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { calls += 's'; return hipSuccess; }
extern "C" hipError_t hipFree(void *) { calls += 'f'; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipMalloc(void **p, size_t size) {
    if (size > most || (held_by && size > held_by())) { calls += 'x'; return hipErrorOutOfMemory; }
    calls += 'm';
    *p = reinterpret_cast<void *>(next_address);
    next_address += size;
    return hipSuccess;
}
static int failures = 0;
namespace zhip {
zhip_result fail(const Dispatch &d, zhip_result code, const char *, ...) {
    failures += d.err && d.err_cap;
    return code;
}
}

static void check(bool ok, const char *what) {
    if (!ok) { printf("FAILED: %s (%s)\n", what, calls.c_str()); exit(1); }
}
static bool called(const char *what) {
    const bool same = calls == what;
    if (same) calls.clear();
    return same;
}

int main() {
    const uint64_t MB = 1u << 20;
    char err[64];
    Dispatch d;
    d.err = err;
    d.err_cap = sizeof err;
    Workspace w;
    check(w.reserve(d, 5) == ZHIP_OK && w.bytes == 8 * MB && w.used && called("sm"), "the first use");
    check(w.reserve(d, 8 * MB) == ZHIP_OK && called(""), "what is there");
    check(w.reserve(d, 8 * MB + 1) == ZHIP_OK && w.bytes == 16 * MB && called("sfm"), "more");

    // During a capture: what is there, and no call that would end it.
    uint8_t *const data = w.data;
    w.kept = true;
    check(w.reserve(d, 16 * MB) == ZHIP_OK && w.data == data && called(""), "kept: what is there");
    check(w.reserve(d, 16 * MB + 1) != ZHIP_OK && failures == 1 && w.data == data && w.bytes == 16 * MB && called(""), "kept: more");
    check(!w.reserve_quietly(d, 17 * MB) && failures == 1 && w.refused == ~0ull && called(""), "kept: more, quietly");
    w.kept = false;

    // Memory is short: one launch of a step asks, and waits for those before it; the others of that size or more do without.
    most = 16 * MB;
    PackedCopy packed;
    packed.room = &w;
    packed.kind = PackedCopy::bf16;
    packed.rows = 512;
    packed.k = 17 * 1024;
    check(!packed.reserve(d) && failures == 1 && called("sfx"), "short");
    check(!packed.reserve(d) && called(""), "still short");
    RoundedCopy rounded;
    rounded.room = &w;
    rounded.rows = 512;
    rounded.k = 30 * 1024;  // 15 MB and their scales
    check(!rounded.reserve(d) && called("sx"), "a little less");
    check(!rounded.reserve(d) && !packed.reserve(d) && called(""), "both still short");
    rounded.k = 1024;
    check(rounded.reserve(d) == w.data && w.bytes == 8 * MB && called("sm"), "what there is room for");
    w.refused = ~0ull;
    most = ~0ull;
    check(packed.reserve(d) && w.bytes == 24 * MB && failures == 1 && called("sfm"), "memory is there again");

    // The most a place holds, of both planes of a split; nowhere to put them.
    packed.k = 65536;
    check(packed.reserve(d) && w.bytes == 64 * MB && called("sfm"), "one plane of the most");
    packed.kind = PackedCopy::f16_split;
    packed.k = 32768;
    check(packed.reserve(d) && called(""), "two planes of the most");
    packed.k = 32768 + 8;
    check(!packed.reserve(d) && called(""), "two planes of more");
    packed.kind = PackedCopy::bf16;
    packed.k = 65536 + 8;
    check(!packed.reserve(d) && called(""), "one plane of more");
    rounded.k = 128 * 1024;
    check(!rounded.reserve(d) && called(""), "a rounding of more");
    rounded.room = nullptr;
    rounded.k = 32;
    check(!rounded.reserve(d) && called(""), "no place");

    // Short of memory for a workspace or a buffer: what the places hold is given back for it, as much as it takes.
    most = 1ull << 40;
    Workspace places[kSpareWorkspaces], work;
    work.spare = places;
    for (Workspace &p : places) check(p.reserve(d, 64 * MB) == ZHIP_OK && called("sm"), "places");
    const uint64_t all = 100 * MB;
    held_by = [&] { return all - places[0].bytes / 2 - places[1].bytes / 2; };  // (what hipMalloc has left)
    void *p = nullptr;
    check(allocate(&p, 30 * MB, nullptr, places) == hipSuccess && p && called("m"), "room enough");
    check(allocate(&p, 60 * MB, nullptr, places) == hipSuccess && called("xsfm") && !places[0].data && places[1].bytes == 64 * MB, "one given back");
    check(places[0].reserve(d, 64 * MB) == ZHIP_OK && called("sm"), "there again");
    check(allocate(&p, 101 * MB, nullptr, places) == hipErrorOutOfMemory && called("xsfxsfx") && !places[0].data && !places[1].data, "both, and not enough");
    check(allocate(&p, 101 * MB, nullptr, places) == hipErrorOutOfMemory && called("x"), "nothing to give");
    check(places[1].reserve(d, 64 * MB) == ZHIP_OK && called("sm") && work.reserve(d, 90 * MB) == ZHIP_OK && called("sxsfm") && !places[1].data, "a workspace");
    check(allocate(&p, 101 * MB, nullptr, nullptr) == hipErrorOutOfMemory && called("x"), "without any");
    held_by = nullptr;
    work.release();
    calls.clear();

    w.release();
    check(!w.data && w.bytes == 0 && called("f"), "given back");
    w.data = data;
    w.bytes = 4;
    w.fixed = true;
    check(w.reserve(d, 4) == ZHIP_OK && w.reserve(d, 5) != ZHIP_OK && failures == 2 && called(""), "not its own");
    printf("ok\n");
}
"""


def test_workspace_under_a_capture_and_short_memory(tmp_path):
    source, program = tmp_path / "workspace.cpp", tmp_path / "workspace"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, "-o", str(program), str(source),
                    os.path.join(CSRC, "workspace.cpp")], check=True)
    r = subprocess.run([str(program)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
