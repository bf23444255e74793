"""The rule that chooses tiles and cuts for products whose tokens' side is in three parts (csrc/qmk_hybrid_tiles.h, compiled for the host): the GPU tests of the products
reach every kind, cut and not, and a cut has room for its tickets and sums at any size."""
import random
import subprocess

import pytest

from conftest import ROOT
from test_gpu_hybrid_products import LENGTHS, SHAPES
from test_hybrid_tiles import products

DRIVER = """
#include <stdio.h>
#include "qmk_hybrid_tiles.h"
using namespace qmk::hybrid;
int main() {
  int M, N, K, groups;
  while (scanf("%d %d %d %d", &M, &N, &K, &groups) == 4) {
    const PartTiles t = choose_part_tiles(M, N, K, groups);
    printf("%d %d %d %d %d %d\\n", t.kind, t.splits, kPartCosts[t.kind].bm, kPartCosts[t.kind].bn, kMaxTickets, kPartialUnits);
  }
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    folder = tmp_path_factory.mktemp("part_tiles")
    (folder / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'qimeng-megakernel_amd' / 'csrc'}", "-o", str(folder / "driver"), str(folder / "driver.cpp")], check=True)

    def run(sizes):
        out = subprocess.run([str(folder / "driver")], input="".join("%d %d %d %d\n" % s for s in sizes), capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def test_the_gpu_tests_reach_every_kind(choose):
    sizes = {(M, N, K, groups) for shape in SHAPES.values() for n in LENGTHS for M, N, K, groups, _, may in products(shape, n) if may and K > 64 and K % 64 == 0}
    found = {(kind, splits > 1) for kind, splits, *_ in choose(sorted(sizes))}
    assert {kind for kind, _ in found} == {0, 1, 2} and {(0, True), (1, True)} <= found


def test_what_is_cut_has_room(choose):
    rng = random.Random(2)
    sizes = [(int(2 ** rng.uniform(0, 13)), 16 * int(2 ** rng.uniform(0, 14)), 64 * int(2 ** rng.uniform(1, 8.5)), rng.choice((1, 1, 5))) for _ in range(4000)]
    for (M, N, K, groups), (_, splits, bm, bn, tickets, units) in zip(sizes, choose(sizes)):
        tiles = -(-M // bm) * -(-N // bn) * groups
        assert splits == 1 or (tiles <= tickets and tiles * splits * bm * bn // 4 <= units and K // splits >= 256)
