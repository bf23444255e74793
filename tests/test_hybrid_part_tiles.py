"""The rule that chooses tiles and cuts for products whose tokens' side is in three parts (csrc/qmk_hybrid_tiles.h, compiled for the host): the GPU tests of the products
reach every kind with every cut that a shape of the registry takes it with, and a cut has room for its tickets and sums at any size."""
import random
import subprocess

import pytest

from conftest import ROOT
from qimeng_megakernel_amd import registry
from test_gpu_hybrid_products import LENGTHS, LONG, LONG_LENGTHS, SHAPES
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


def pairs(choose, portions):
    """{(kind, cuts)} of the products of (shape, tokens) whose tokens' side is in parts."""
    sizes = {(M, N, K, groups) for shape, n in portions for M, N, K, groups, _, may in products(shape, n) if may and K > 64 and K % 64 == 0}
    return {(kind, cuts) for kind, cuts, *_ in choose(sorted(sizes))}


def test_the_gpu_tests_reach_every_kind_and_cut(choose):
    tested = pairs(choose, [(shape, n) for shape in SHAPES.values() for n in LENGTHS] + [(LONG, n) for n in LONG_LENGTHS])
    shapes = [registry.shape_of(name) for name, (family, *_) in registry.MODELS.items() if family is registry.HYBRID]
    used = pairs(choose, [(shape, n) for shape in shapes for n in (*range(2, 700), *range(700, 4097, 31))])
    assert len(shapes) >= 4 and used == {(0, 1), (0, 2), (0, 4), (0, 8), (1, 1), (1, 2), (1, 4), (2, 1), (2, 2), (2, 4)} and used <= tested


def test_what_is_cut_has_room(choose):
    rng = random.Random(2)
    sizes = [(int(2 ** rng.uniform(0, 13)), 16 * int(2 ** rng.uniform(0, 14)), 64 * int(2 ** rng.uniform(1, 8.5)), rng.choice((1, 1, 5))) for _ in range(4000)]
    for (M, N, K, groups), (_, splits, bm, bn, tickets, units) in zip(sizes, choose(sizes)):
        tiles = -(-M // bm) * -(-N // bn) * groups
        assert splits == 1 or (tiles <= tickets and tiles * splits * bm * bn // 4 <= units and K // splits >= 256)
