"""Which launch of the K formats' int8 multiply a step takes (zllm_amd/csrc/matmul_kquant_launch.h), on the CPU, built with g++."""
import os
import subprocess

import pytest

from test_gpu_check import KQUANT_HALVES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zllm_amd", "csrc")

# Each line "type rows n blocks": the launch's token tiles, row groups and split; "type 0 0 blocks": every launch that steps of
# 1 ... 512 tokens over up to 1100 row groups take.
PROGRAM = r"""
#include "matmul_kquant_launch.h"
#include <cstdio>
#include <set>
using namespace zhip;
int main() {
    int type;
    unsigned rows, n, blocks;
    while (scanf("%d %u %u %u", &type, &rows, &n, &blocks) == 4) {
        const KquantCosts c = kquant_costs(type);
        std::set<int> taken;
        if (rows) taken.insert(kquant_launch(c, rows, n, 256 * blocks, 256));
        else
            for (unsigned groups = 1; groups <= 1100; groups++)
                for (unsigned tokens = 1; tokens <= 512; tokens += 31) taken.insert(kquant_launch(c, tokens, 32 * groups, 256 * blocks, 256));
        for (int i : taken) printf("%u,%u,%u ", kKquantLaunches[i].tiles, kKquantLaunches[i].groups, kKquantLaunches[i].split);
        printf("\n");
    }
}
"""


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    folder = tmp_path_factory.mktemp("kquant_launch")
    source, program = folder / "launch.cpp", folder / "launch"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, "-o", str(program), str(source)], check=True)

    def ask(lines):
        out = subprocess.run([str(program)], input="\n".join(" ".join(map(str, l)) for l in lines), capture_output=True, text=True, check=True, timeout=100).stdout
        return [{tuple(map(int, l.split(","))) for l in line.split()} for line in out.splitlines()]

    return ask


def test_launches_of_two_parts_of_k(launches):
    """The steps that test_matmul_kquant_int8_halves_of_k runs: a wave a part over the small matrix, and over the tall one every
    launch of two parts a wave in every number of blocks that any step takes it in."""
    n, times, blocks, steps = KQUANT_HALVES
    for t in (3, 4, 5, 6):
        for b in blocks:
            small, tall = (launches([(t, count, rows, b) for _, count in steps]) for rows in (n, n * times))
            assert {split for taken in small for _, _, split in taken} == {4}, (t, b)
            ran = {l for taken in tall for l in taken}
            assert {l for l in ran if l[2] == 2} == {l for l in launches([(t, 0, 0, b)])[0] if l[2] == 2}, (t, b)
            assert 1 in {split for _, _, split in ran}


def test_launches_by_format_and_blocks(launches):
    """One and two blocks a row have no step with one token tile a workgroup and two parts a wave, and Q4_K's of one block and Q5_K's of one and two none
    of two parts at all; a few of the costs' lines."""
    two = {(t, b): {l[:2] for l in launches([(t, 0, 0, b)])[0] if l[2] == 2} for t in (3, 4, 5, 6) for b in (1, 2, 3, 5, 9)}
    assert [two[3, b] for b in (1, 2, 3, 5, 9)] == [{(2, 2)}] * 4 + [{(2, 2), (1, 4)}]
    assert [two[4, b] for b in (1, 2, 3, 5, 9)] == [set(), {(2, 4)}] + [{(2, 4), (1, 4)}] * 3
    assert [two[5, b] for b in (1, 2, 3, 5, 9)] == [set(), set(), {(1, 4)}] + [{(2, 4), (1, 4)}] * 2
    assert [two[6, b] for b in (1, 2, 3, 5, 9)] == [{(2, 2)}] * 2 + [{(2, 2), (1, 4)}] * 3
    steps = [(4, 64, 28672, 16), (4, 64, 4096, 16), (4, 512, 28672, 16), (6, 64, 24576, 12), (6, 256, 19456, 10), (3, 32, 28672, 16)]
    assert [launches([s])[0] for s in steps] == [{(2, 4, 2)}, {(1, 1, 4)}, {(2, 4, 1)}, {(2, 2, 2)}, {(2, 2, 2)}, {(1, 4, 2)}]
