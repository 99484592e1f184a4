// Which launch of matmul_kquant_i8.hip a step takes: host code alone.
#pragma once

#include "common.h"

namespace zhip {

// A workgroup's token tiles and row groups of 32, and the waves of a row group that k is split over (S).
struct KquantLaunch { uint32_t tiles, groups, split; };
constexpr int kKquantLaunchCount = 11;
constexpr KquantLaunch kKquantLaunches[kKquantLaunchCount] = {{1, 1, 4}, {1, 2, 4}, {2, 1, 4}, {2, 2, 4}, {4, 2, 4}, {1, 4, 1}, {2, 4, 1}, {4, 4, 1}, {1, 4, 2}, {2, 4, 2}, {2, 2, 2}};

// Which launch takes a step; the bits are the same. Workgroups that walk a part of k each (S = 4), or two with four row groups
// (S = 2), have a CU to themselves: a launch of w a CU takes w times one's time. Those that walk all of it (S = 1), or half of it for
// two row groups, share a CU two at a time, and a pair takes less than twice a lone one's time: an odd one out costs `lone`, a pair `pair`. In k the
// first kinds' time grows like blocks + 3 (the exchange), the third's like blocks + 2. In units of such a
// time, fitted to steps of 16 ... 512 tokens over sixteen matrices of 1024 x 3072 ... 28672 x 4096 and 4096 x 14336, every
// launch of the list on each of them: the rule's launch is within 0.2 % (Q5_K 0.9 %, Q6_K 0.6 %) of the fastest one in the mean, and the launches
// of S = 2 take 0.89 (Q3_K), 0.92, 0.92 and 0.91 of the time of those they came in place of. (A line
// at a number of workgroups, as here before, lost 1.6 % / 6.2 % / 2.7 % / 1.8 % of Q4_K's / Q5_K's / Q6_K's / Q3_K's time, and where a
// last round was nearly empty 30 - 80 %: 96 x 19456 x 2560 Q4_K 34.9 -> 20.5 us, Q5_K 40.6 -> 22.5, Q3_K 25.1 -> 19.0; Q5_K
// 512 x 12288 x 2560 63.4 -> 55.9, 64 x 28672 x 4096 Q4_K 33.1 -> 31.6.)
struct KquantCosts {
    uint32_t parts[5];   // launches 0 .. 4
    SharedCu whole[3];   // 5 .. 7 (of two planes, four tiles' closed sums do not fit the registers)
    uint32_t halves[2];  // 8, 9
    SharedCu halves2;    // 10
    // (0: none, or never the cheapest)
    constexpr bool has(int i) const { return (i < 5 ? parts[i] : i < 8 ? whole[i - 5].lone : i < 10 ? halves[i - 8] : halves2.lone) != 0u; }
};
// Of Q3_K ... Q6_K.
constexpr KquantCosts kquant_costs(int type) {
    return type == 3 ? KquantCosts{{19, 24, 22, 31, 42}, {{51, 73}, {67, 90}, {98, 118}}, {45, 0}, {32, 46}}
        : type == 4 ? KquantCosts{{14, 19, 18, 29, 0}, {{39, 56}, {50, 71}, {0, 0}}, {32, 38}, {0, 0}}
        : type == 5 ? KquantCosts{{13, 17, 19, 26, 40}, {{32, 47}, {51, 79}, {0, 0}}, {26, 41}, {0, 0}}
                    : KquantCosts{{17, 26, 21, 31, 43}, {{53, 74}, {66, 91}, {0, 0}}, {43, 0}, {40, 44}};
}

inline int kquant_launch(const KquantCosts &c, uint32_t rows, uint32_t n, uint32_t k, uint32_t compute_units) {
    const uint64_t cus = compute_units, row_groups = (n + 31u) / 32u, blocks = k / 256u;
    uint64_t least = ~0ull;
    int best = 0;
    for (int i = 0; i < kKquantLaunchCount; i++) {
        if (!c.has(i)) continue;
        const KquantLaunch &l = kKquantLaunches[i];
        const uint64_t workgroups = (row_groups + l.groups - 1u) / l.groups * ((rows + 32u * l.tiles - 1u) / (32u * l.tiles)), rounds = (workgroups + cus - 1u) / cus;
        const uint64_t cost = i < 5 ? c.parts[i] * rounds * (blocks + 3u) : i < 8 ? c.whole[i - 5].of(workgroups, cus) * (blocks + 2u) : i < 10 ? c.halves[i - 8] * rounds * (blocks + 3u)
                                                                                                                          : c.halves2.of(workgroups, cus) * (blocks + 3u);
        if (cost < least) least = cost, best = i;
    }
    return best;
}

}  // namespace zhip
