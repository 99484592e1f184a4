"""The second thread of long reads (zllm_amd/csrc/handover.h) on the CPU, built with g++: pieces whose
flags a third thread sets in the GPU's place, or never does, as after a device error."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zllm_amd", "csrc")

PROGRAM = r"""
#include "handover.h"
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace zhip;
using std::chrono::milliseconds;

static void check(bool ok, const char *what) {
    if (!ok) { printf("FAILED: %s\n", what); exit(1); }
}

struct Job {
    std::vector<uint8_t> src, dst;
    std::vector<uint64_t> flags;
    Handover h;
    // (what the flags hold from before differs from the ticket in the upper half alone)
    Job(uint64_t size, uint64_t piece, uint64_t ticket) : src(size), dst(size, 0xee), flags((size + piece - 1) / piece, ticket) {
        ticket += 1ull << 32;
        h = Handover{dst.data(), src.data(), size, piece, flags.data(), ticket};
    }
    // Piece p as the GPU leaves it.
    void bring(uint64_t p) {
        for (uint64_t i = p * h.piece; i < std::min(h.size, (p + 1) * h.piece); i++) src[i] = (uint8_t)(i * 7 + h.ticket);
        __atomic_store_n(flags.data() + p, h.ticket, __ATOMIC_RELEASE);
    }
    bool whole(uint64_t first, uint64_t last) const {
        for (uint64_t i = first; i < last; i++) if (dst[i] != (uint8_t)(i * 7 + h.ticket)) return false;
        return true;
    }
    bool untouched(uint64_t first) const {
        for (uint64_t i = first; i < h.size; i++) if (dst[i] != 0xee) return false;
        return true;
    }
};

struct Thread : HandoverThread {
    bool waits_for(uint64_t p) const { return taken_.load() >> 32 == p + 1; }
};

int main() {
    Thread t;
    // `come` of ten pieces arrive, the thread copies those (nobody else does) and waits for one more, which
    // the caller takes back with the others or not at all: either way the wait for the thread ends.
    for (uint64_t come : {0, 1, 5, 9})
        for (bool back : {false, true}) {
            Job j(10 * 1000 - 3, 1000, 77);
            t.start(j.h);
            for (uint64_t p = 0; p < come; p++) j.bring(p);
            while (!t.waits_for(come)) std::this_thread::sleep_for(milliseconds(1));
            if (back) {
                for (uint64_t p = come + 1; p < 10; p++) check(t.take() == p, "a piece nobody has");
                check(t.take() == come, "the thread's piece");
                check(t.take() == HandoverThread::kNone, "nothing is left");
                for (uint64_t p = come; p < 10; p++) j.bring(p);
                std::this_thread::sleep_for(milliseconds(20));
            }
            t.finish();
            check(j.whole(0, come * 1000) && j.untouched(come * 1000), "what had arrived before, and no more");
        }
    // All of them, from a third thread, copied by the two of them; a late caller, one that is as quick, and one piece alone.
    uint32_t seed = 1;
    auto random = [&](uint32_t n) { return (seed = seed * 1664525u + 1013904223u) >> 8, (seed >> 8) % n; };
    for (uint32_t turn = 1; turn <= 400; turn++) {
        const uint64_t piece = 16 + random(5000), size = turn % 9 == 0 ? 1 + random((uint32_t)piece) : 1 + random(60000);
        Job j(size, piece, turn);
        t.start(j.h);
        std::thread gpu([&] {
            for (uint64_t p = 0; p < j.h.pieces(); p++) {
                if (turn % 5 == 0) std::this_thread::sleep_for(std::chrono::microseconds(50));
                j.bring(p);
            }
        });
        if (turn % 3 == 0) std::this_thread::sleep_for(std::chrono::microseconds(random(300)));
        for (uint32_t p; (p = t.take()) != HandoverThread::kNone;) {
            while (!j.h.arrived(p)) pause_cpu();
            j.h.copy(p);
        }
        t.finish();
        check(j.whole(0, size), "every byte of every piece");
        gpu.join();
    }
    printf("ok\n");
}
"""


def test_handover_thread_ends_whatever_arrives(tmp_path):
    source, program = tmp_path / "handover.cpp", tmp_path / "handover"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-pthread", "-I", CSRC, "-o", str(program), str(source)], check=True)
    r = subprocess.run([str(program)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
