"""The rules that choose a prefill product's tiles (csrc/qmk_hybrid_tiles.h, compiled for the host): what the GPU tests of the products reach, and properties that
hold for any size."""
import random
import subprocess

import pytest

from conftest import ROOT
from test_gpu_hybrid_products import LENGTHS, SHAPES

KINDS = ("Tiles64", "Wide256", "Wide64", "Turns96", "Turns128", "Tall192", "Tall256", "Turns192", "Turns256", "Tiles32", "Few64", "Few32")
DRIVER = """
#include <stdio.h>
#include "qmk_hybrid_tiles.h"
using namespace qmk::hybrid;
int main() {
  int M, N, K, groups, streams, cut;
  while (scanf("%d %d %d %d %d %d", &M, &N, &K, &groups, &streams, &cut) == 6) {
    const RegisterTiles r = choose_register_tiles(M, N, K, groups, cut);
    const int kind = K % 64 ? -1 : choose_tiles(M, N, K, groups, streams);
    printf("%d %d %d %d %d %d %d\\n", kind, kind < 0 ? 1 : kTileCosts[kind].bm, kind < 0 ? 1 : kTileCosts[kind].bn, kind < 0 ? 1 : kTileCosts[kind].bk, choose_part_tiles(M, N, K, groups).splits,
           r.large, r.splits);
  }
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    folder = tmp_path_factory.mktemp("tiles")
    (folder / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'qimeng-megakernel_amd' / 'csrc'}", "-o", str(folder / "driver"), str(folder / "driver.cpp")], check=True)

    def run(sizes):
        """(kind, its rows of tokens, of weights, its columns, cuts of parts, whether register tiles are large, their cuts) of (M, N, K, groups, whether the
        epilogue moves the residual's streams, whether there is an fp32 side)."""
        text = "".join("%d %d %d %d %d %d\n" % s for s in sizes)
        out = subprocess.run([str(folder / "driver")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def products(shape, n):
    """(M, N, K, groups, whether the epilogue moves the residual's streams, whether its tokens' side may be in parts) of every product of a portion of n
    tokens from a request's start."""
    D, S, found = shape.width_s, int(not shape.plain), []
    for e in shape.entries:
        l = e.shape
        if e.type == "join":
            found.append((n, D, 2 * D, 1, 0, True))
        if e.type in ("join", "final"):
            continue
        if e.type == "wkv":
            found += [(n, max(l.mix_width, l.rank_s), D, 5, 0, True), (n, l.mix_width, l.rank_s, 1, 0, False)]
        else:
            found.append((n, l.in_rows, D, 1, 0, True))
        if e.type == "rglru":
            found.append((n, 2 * l.block_s, l.block_s, l.blocks, 0, False))
        elif e.type == "latent_attention":
            found += [(n, l.heads * l.dim_s, l.rank_s, 1, 0, False), (l.heads * l.v_s, n, l.rank_s, 1, 0, False)]
        elif e.type in ("delta", "gla"):
            found.append((n, l.heads * l.dim_s, l.rank_s, 1, 0, False))
            if e.type == "delta":
                found.append((n, l.mix_width, l.gate_rank_s, 1, 0, False))
        found.append((n, D, l.mix_width, 1, S, True))
        ff = (16 * -(-e.ff // 16)) if e.ff else 0
        if ff:
            found += [(n, 2 * ff, D, 1, 0, True), (n, D, ff, 1, S, True)]
    return found + [(n, shape.vocab_s, D, 1, 0, True)]


def test_the_gpu_tests_reach_every_kind_of_tile(choose):
    tiles, parts, register = {}, set(), set()
    for name, shape in SHAPES.items():
        for n in LENGTHS:
            sizes = products(shape, n)
            for (M, N, K, *_), (kind, bm, bn, *_) in zip(sizes, choose([s[:5] + (0,) for s in sizes])):
                if kind >= 0:
                    tiles.setdefault(KINDS[kind], set()).update(side for side, over in (("tokens", M % bm), ("rows", N % bn)) if over)
            for (M, N, K, *_, may), (*_, cuts, large, small_cuts) in zip(sizes, choose([s[:5] + (1,) for s in sizes])):
                if may and K > 64 and K % 64 == 0:
                    parts.add(cuts)
                elif K > 64:
                    register.add("large" if large else small_cuts)
    # with tokens and rows of weights that they do not divide (rows come in sixteens, which Few32 and Few64 always divide)
    assert tiles == {kind: {"tokens", "rows"} if "Few" not in kind else {"tokens"} for kind in KINDS}
    assert parts == {1, 2, 4, 8} and register == {"large", 1, 2, 4, 8}


def test_rules_hold_for_any_size(choose):
    rng = random.Random(1)
    sizes = [(int(2 ** rng.uniform(0, 13)), 16 * int(2 ** rng.uniform(0, 14)), 16 * int(2 ** rng.uniform(0, 10.5)), rng.choice((1, 1, 5, 10)), rng.randint(0, 1), rng.randint(0, 1)) for _ in range(4000)]
    for (M, N, K, groups, _, fp32), (kind, bm, bn, bk, cuts, large, small_cuts) in zip(sizes, choose(sizes)):
        if kind >= 0:
            assert K % bk == 0
        # what is cut has room for its tickets and sums, and every part has columns of its own
        for tiles, per, c in ((-(-M // 32) * -(-N // 128) * groups, 32 * 128, cuts), (-(-M // 64) * -(-N // 64) * groups, 64 * 64, small_cuts)):
            if c > 1:
                assert tiles <= 512 and tiles * c * per // 4 <= 256 * 128 * 128 // 4 and K // c >= 256
        assert fp32 or small_cuts == 1
        assert not large or small_cuts == 1


#: us by kind of (tokens, rows of weights, columns, whether the epilogue moves the residual's streams): a launch in a whole portion of a shape that has the product, all of
#: whose products take the kind (so weights and streams come from memory); mean over its launches on one MI355X, the three fastest kinds
MEASURED = [
    ((43, 2048, 6144, 1), {"Few32": 15.0, "Few64": 20.9, "Tiles32": 22.8}),
    ((43, 2048, 2048, 1), {"Few32": 8.7, "Few64": 10.4, "Tiles32": 12.8}),
    ((43, 5696, 2048, 0), {"Tiles32": 10.6, "Few64": 11.8, "Tiles64": 13.5}),
    ((43, 12288, 2048, 0), {"Tiles64": 15.2, "Tiles32": 16.7, "Wide64": 18.4}),
    ((128, 2048, 8192, 1), {"Few64": 26.9, "Tiles32": 30.7, "Tiles64": 41.5}),
    ((200, 2048, 6144, 1), {"Few64": 28.2, "Tiles64": 32.1, "Wide64": 46.7}),
    ((260, 6144, 2048, 0), {"Tiles64": 19.9, "Turns128": 22.1, "Turns96": 24.2}),
    ((400, 5696, 2048, 0), {"Turns128": 20.4, "Turns96": 20.8, "Wide64": 25.5}),
    ((520, 2048, 6144, 1), {"Tiles64": 41.9, "Wide64": 47.0, "Turns128": 52.4}),
    ((520, 12288, 2048, 0), {"Wide256": 31.8, "Turns128": 36.2, "Wide64": 44.2}),
    ((1024, 2048, 6144, 1), {"Wide64": 54.6, "Turns96": 56.5, "Tiles64": 64.8}),
    ((1531, 2048, 2048, 1), {"Turns96": 33.6, "Turns128": 36.8, "Wide64": 42.6}),
    ((1531, 2048, 8192, 1), {"Turns96": 72.6, "Turns128": 84.6, "Tall192": 100.7}),
    ((1531, 16384, 2048, 0), {"Tall256": 94.9, "Wide256": 100.1, "Turns192": 101.6}),
    ((1531, 5696, 2048, 0), {"Tall192": 56.4, "Turns192": 56.5, "Tall256": 58.5}),
    ((2048, 2048, 2048, 1), {"Turns128": 42.8, "Tall192": 49.1, "Turns96": 52.4}),
    ((2048, 2048, 2048, 0), {"Turns128": 25.3, "Tall192": 28.0, "Wide64": 32.3}),
    ((2048, 2048, 8192, 1), {"Turns128": 93.6, "Tall192": 103.5, "Tall256": 121.5}),
    ((2048, 12288, 2048, 0), {"Tall256": 94.5, "Wide256": 99.8, "Turns256": 117.7}),
    ((2048, 16384, 2048, 0), {"Turns256": 123.2, "Tall256": 125.4, "Wide256": 134.2}),
    ((3000, 2048, 2048, 1), {"Tall192": 61.4, "Tall256": 67.3, "Turns96": 67.8}),
    ((3000, 2048, 8192, 0), {"Tall192": 97.8, "Tall256": 111.5, "Wide256": 115.4}),
    ((4096, 2048, 8192, 0), {"Wide256": 131.6, "Tall256": 132.1, "Turns192": 161.0}),
    ((4096, 2048, 8192, 1), {"Wide256": 166.2, "Tall256": 172.4, "Turns128": 207.1}),
    ((4096, 16384, 2048, 0), {"Turns256": 248.9, "Tall256": 253.5, "Wide256": 273.3}),
]


def test_choices_where_kinds_were_measured(choose):
    got = choose([(M, N, K, 1, streams, 0) for (M, N, K, streams), _ in MEASURED])
    slower = {size: us.get(KINDS[kind], float("inf")) / min(us.values()) for (size, us), (kind, *_) in zip(MEASURED, got)}
    assert max(slower.values()) < 1.04, slower
