"""The rule that picks the sort of a build's keys (gprt_amd/csrc/build_rule.hpp), compiled and asked on the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <vector>
#include "gprt_amd/csrc/build_rule.hpp"
int main() {  // lines of: tile size, number of {meshes, primitives} pairs, the pairs
  unsigned tile, parts;
  while (std::scanf("%u %u", &tile, &parts) == 2) {
    std::vector<unsigned> sizes;
    for (unsigned p = 0, count, n; p < parts && std::scanf("%u %u", &count, &n) == 2; ++p) sizes.insert(sizes.end(), count, n);
    std::printf("%u\\n", gprt::rank_groups((unsigned)sizes.size(), tile, [&](unsigned m) { return sizes[m]; }));
  }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    at = tmp_path_factory.mktemp("rule")
    (at / "rule.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", ROOT, "-o", str(at / "rule"), str(at / "rule.cpp")], check=True)

    def ask(parts, tile=2048):
        line = " ".join([str(tile), str(len(parts))] + ["%d %d" % p for p in parts])
        return int(subprocess.run([str(at / "rule")], input=line, capture_output=True, text=True, check=True).stdout)

    return ask


@pytest.mark.parametrize("parts", [[(1, 1)], [(1, 64)], [(1, 65)], [(1, 2048)], [(1, 2049)], [(1, 11585)], [(1, 11586)],
                                   [(131072, 32)], [(131072, 8), (1, 11000)], [(65536, 8)], [(4096, 64)],
                                   [(2_000_000, 8)], [(3_000_000, 4)], [(1, 8000), (4000, 8)], [(1, 2000), (500, 8)],
                                   [(1, 600), (2000, 64)]])
def test_ranks_launch_what_has_keys(rule, parts):
    """Workgroups of 1,024 threads for 64 keys each: they cover every tile, stay far below the 2^32 threads
    of a launch, and few of them are idle."""
    groups = rule(parts)
    tiles = sum(c * -(-n // 2048) for c, n in parts)
    busy = sum(c * -(-n // 64) for c, n in parts)
    largest = max(n for _, n in parts)
    if groups:
        assert groups * 64 >= min(largest, 2048)
        assert tiles * groups * 1024 < 2**32
        assert tiles * groups - busy <= 16 * tiles + 8192


def test_which_builds_take_ranks(rule):
    assert rule([(1, 11585)]) == 32 and rule([(1, 11586)]) == 0
    assert rule([(4096, 64)]) == 1 and rule([(1000, 8), (1, 150)]) == 3
    assert rule([(1, 2000), (500, 8)]) == 32 and rule([(1, 2000), (1000, 8)]) == 0
    assert rule([(65536, 8)]) == 1 and rule([(3_000_000, 4)]) == 0
