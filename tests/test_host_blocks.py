"""CPU tests of the block order of the bf16 kernels (csrc/ltr_blocks.h: the arithmetic that the kernels run, compiled with the host
compiler): every block of a launch exactly once, a pair's blocks on one XCD, and the order on both sides of the grid's limits."""
import os
import shutil
import subprocess

import pytest

import lightron_amd as la

CSRC = os.path.join(os.path.dirname(la.__file__), "csrc")
PROGRAM = r"""
#include "ltr_blocks.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
// pairs items inner group -> the grid, "ok" and the largest number of pairs of an XCD that are begun and not finished at a time;
// pairs blocks_per_pair slots "group" -> pair_group of uneven blocks and the pairs of the last group
int main(int argc, char **argv) {
    const long long pairs = atoll(argv[1]), items = atoll(argv[2]), inner = atoll(argv[3]);
    if (argv[4][0] == 'g') {
        const long long n = pairs / 8, group = pair_group(pairs, items, (int)inner, true);
        printf("%lld %lld\n", group, n - (n - 1) / group * group);
        return 0;
    }
    const BlockGrid g = block_grid(pairs, items, inner, atoll(argv[4]));
    printf("%d %u %u %u ", g.map.group, g.x, g.y, g.z);
    if (g.y > GRID_YZ_MAX || g.z > GRID_YZ_MAX) return printf("too large\n"), 1;
    std::vector<unsigned char> seen(pairs * items * inner);
    std::vector<long long> left(pairs, items * inner);
    long long open[8] = {}, most = 0, id = 0, blocks = 0, order[8] = {};
    for (unsigned z = 0; z < g.z; z++)
        for (unsigned y = 0; y < g.y; y++)
            for (unsigned x = 0; x < g.x; x++, id++) {
                const int xcd = id & 7;
                const BlockItem b = block_item_at(g.map, (int)pairs, x, y, z);
                if (b.order != order[xcd]++) return printf("order\n"), 1;
                if (b.pair >= pairs) continue;
                if (b.pair < 0 || b.item < 0 || b.item >= items || b.sub < 0 || b.sub >= inner) return printf("range\n"), 1;
                if (pairs % 8 == 0 && (b.pair & 7) != xcd) return printf("xcd\n"), 1;
                if (seen[(b.pair * items + b.item) * inner + b.sub]++) return printf("twice\n"), 1;
                blocks++;
                if (left[b.pair] == items * inner) open[xcd]++;
                if (open[xcd] > most) most = open[xcd];
                if (--left[b.pair] == 0) open[xcd]--;
            }
    if (blocks != pairs * items * inner) return printf("missing\n"), 1;
    printf("ok %lld\n", most);
    return 0;
}
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    cxx = os.environ.get("CXX", "g++")
    if not shutil.which(cxx):
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("blocks")
    (d / "blocks.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", CSRC, str(d / "blocks.cpp"), "-o", str(d / "blocks")], check=True)
    return lambda *a: subprocess.run([str(d / "blocks")] + [str(x) for x in a], capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize("pairs,items,inner,group", [
    (8, 1, 1, 1), (8, 5, 4, 1), (40, 7, 1, 5), (40, 7, 2, 3), (104, 18, 1, 7), (56, 9, 4, 4), (24, 46, 2, 3),
    (1, 3, 2, 1), (60, 5, 1, 1), (7, 9, 4, 1), (12, 4, 3, 1),                             # pairs that do not divide among the XCDs
])
def test_every_block_once(blocks, pairs, items, inner, group):
    out = blocks(pairs, items, inner, group)
    assert out[4] == "ok", out
    if pairs % 8 == 0:
        assert out[0] == str(group) and int(out[5]) <= group


@pytest.mark.parametrize("pairs,items,inner,group,used", [
    (8 * 65535, 1, 1, 1, 1), (8 * 65536, 1, 1, 1, 2),                  # as many pairs as places, and one per XCD more
    (1024, 511, 1, 1, 1), (1024, 512, 1, 1, 2),                        # 1024 pairs of 65536 keys in tiles of 128
    (131072, 4, 1, 1, 2), (131072, 3, 2, 1, 1),                        # 131072 pairs of 512 rows
    (136, 5000, 1, 1, 2), (136, 5000, 1, 3, 3), (16, 65535, 1, 1, 2),
    (8, 65535, 1, 1, 1), (8, 65536, 1, 1, 0), (24, 70000, 1, 2, 0),    # more items than places: linear
])
def test_limits_of_the_grid(blocks, pairs, items, inner, group, used):
    """Past the limit the pairs of an XCD still come a few at a time, not all of them block by block."""
    out = blocks(pairs, items, inner, group)
    assert out[4] == "ok" and out[0] == str(used), out
    assert int(out[5]) <= (used or pairs // 8)


@pytest.mark.parametrize("per_xcd,per_pair,slots,group", [
    (3, 46, 32, 3), (5, 40, 32, 3), (10, 24, 32, 5), (13, 28, 32, 5), (8, 22, 32, 4), (10, 63, 64, 5),       # not 2+1, 2+2+1, 4+4+2, 4+4+4+1, 3+3+2
    (33, 3, 32, 17), (60, 3, 32, 20), (15, 12, 32, 5), (6, 20, 32, 3), (28, 6, 32, 10), (7, 18, 32, 4), (9, 12, 32, 5),   # 1.3 - 1.9 rounds stay
    (1, 10, 32, 1), (8, 8, 32, 8), (24, 8, 32, 8), (32, 16, 32, 4), (16, 64, 32, 1), (16, 200, 32, 1), (4, 12, 96, 4),
])
def test_groups_of_pairs(blocks, per_xcd, per_pair, slots, group):
    assert blocks(8 * per_xcd, per_pair, slots, "group")[0] == str(group)


def test_the_last_group_is_not_a_small_one(blocks):
    """It would end the launch with its own long blocks alone."""
    for per_xcd in (1, 2, 3, 5, 6, 7, 8, 10, 11, 13, 16, 24, 32, 60):
        for per_pair, slots in ((8, 32), (18, 32), (24, 32), (30, 64), (46, 32), (12, 96), (64, 32), (200, 32)):
            group, last = (int(x) for x in blocks(8 * per_xcd, per_pair, slots, "group"))
            assert group == per_xcd or last * per_pair >= 1.4 * slots or last >= 0.7 * group, (per_xcd, per_pair, slots, group, last)
