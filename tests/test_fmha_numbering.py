"""The pipelined attention kernel's workgroup numbering, compiled for the CPU from its own header."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile.jl_amd", "csrc")

# Every id gives a (query block, head) of the launch, no two ids the same one, and the divisions of the head are exact.
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "fmha_pipe128_map.h"
int main(int argc, char** argv) {
    const int nqb = atoi(argv[1]), nbh = atoi(argv[2]), H = atoi(argv[3]), group = atoi(argv[4]);
    const bool causal = atoi(argv[5]) != 0;
    if (!mi::fmha::map_exact(nqb, nbh, H)) return printf("not taken\n"), 0;
    const mi::fmha::Map mp = mi::fmha::make_map(nqb, nbh, H, group, causal);
    std::vector<bool> seen((size_t)nqb * nbh);
    for (int64_t id = 0; id < (int64_t)nqb * nbh; ++id) {
        int qb, bh;
        mp.at((unsigned)id, nqb, causal, &qb, &bh);
        if (qb < 0 || qb >= nqb || bh < 0 || bh >= nbh || seen[(size_t)bh * nqb + qb])
            return printf("id %lld -> query block %d, head %d\n", (long long)id, qb, bh), 1;
        seen[(size_t)bh * nqb + qb] = true;
        if (mp.H.div(bh) != (unsigned)(bh / H) || mp.group.div(bh % H) != (unsigned)(bh % H / group)) return printf("head %d\n", bh), 1;
    }
    printf("ok\n");
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("numbering")
    (d / "map.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "map.cpp"), "-o", str(d / "map")], check=True)
    return str(d / "map")


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("nqb,nbh,H,group", [
    (1, 1, 1, 1), (1, 7, 7, 7), (2, 64, 32, 4), (16, 64, 32, 4), (27, 28, 7, 1), (30, 30, 6, 3), (3, 521, 521, 1), (513, 3, 3, 1), (2, 2056, 8, 2),
    # up to 2^24 workgroups, heads that no XCD has to itself
    (101, 100_001, 1, 1), (97, 126_495, 5, 5), (60, 160_003, 1, 1), (20, 700_001, 1, 1), (1, 16_000_001, 1, 1), (30_000, 101, 1, 1), (100, 128_000, 8, 2),
])
def test_every_workgroup_has_a_query_block_of_its_own(program, nqb, nbh, H, group, causal):
    r = subprocess.run([program, str(nqb), str(nbh), str(H), str(group), str(causal)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
