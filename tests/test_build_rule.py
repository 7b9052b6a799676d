"""The rules that pick tile size and sort of a build's keys (gprt_amd/csrc/build_rule.hpp), compiled and asked on the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <vector>
#include "gprt_amd/csrc/build_rule.hpp"
int main() {  // lines of: tile size (0: asks for it), number of {meshes, primitives} pairs, the pairs
  unsigned tile, parts;
  while (std::scanf("%u %u", &tile, &parts) == 2) {
    std::vector<unsigned> sizes;
    for (unsigned p = 0, count, n; p < parts && std::scanf("%u %u", &count, &n) == 2; ++p) sizes.insert(sizes.end(), count, n);
    auto size = [&](unsigned m) { return sizes[m]; };
    const unsigned meshes = (unsigned)sizes.size();
    std::printf("%u\\n", tile ? gprt::rank_groups(meshes, tile, size) : (unsigned)gprt::auto_tile_keys(meshes, size));
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


def test_tile_sizes(rule):
    """Many meshes of a little over 12,288 primitives take two tiles of 8,192 each rather than four of 4,096."""
    assert rule([(300, 12288)], 0) == 4096 and rule([(300, 12289)], 0) == 8192 and rule([(300, 15000)], 0) == 8192
    assert rule([(1, 384 << 10)], 0) == 2048 and rule([(1, (384 << 10) + 1)], 0) == 4096
    assert rule([(1, 768 << 10)], 0) == 4096 and rule([(1, (768 << 10) + 1)], 0) == 8192
    assert rule([(1, (5 << 19) - 1)], 0) == 8192 and rule([(1, 5 << 19)], 0) == 16384
    assert rule([(4000, 50), (1, 4_000_000)], 0) == 2048
