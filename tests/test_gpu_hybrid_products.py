"""The prefill's matrix products over the sizes at which their tiles change (csrc/qmk_hybrid_tiles.h): layers of every mixer at widths and
lengths where every kind of tile is taken, with tokens and rows of weights it does not divide, cut along K or not (test_hybrid_tiles.py
holds that list against the rules), against the plain implementation in 64 bits.

Tolerances as in test_gpu_hybrid.py and, on a plain residual, test_gpu_looped.py: fp32 at rounding level, bf16 at bf16's."""
import functools

import pytest
import torch

import givopel_oracle
import hybrid_oracle as O
from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu

DEVICE = "cuda:0"
TOL = {torch.float32: 2e-5, torch.bfloat16: 4e-2}
TOL_PLAIN = {torch.float32: 4e-5, torch.bfloat16: 8e-2}
MOST = 1540
#: lengths at which some product of some shape changes its tiles, and odd ones
LENGTHS = (2, 16, 40, 63, 65, 129, 200, 257, 520, 1024, 1100, 1290, 1531, MOST)
#: feed-forwards of a size that fills the large tiles, and of one no tile divides; every mixer, with columns in multiples of 64 and not
SHAPES = {
    "large": synthetic.hybrid_shape("a", width=2048, vocab=640, streams=2, ff={"a": 4096}, heads=8, dim=128, rot_dim=64, v_dim=128, rank=256, window=512),
    "ragged": synthetic.hybrid_shape("a", width=1104, vocab=336, streams=3, ff={"a": 1744}, heads=3, dim=80, rot_dim=32, v_dim=112, rank=144, window=77),
    "recurrent": synthetic.hybrid_shape("rw", width=2112, vocab=336, streams=2, ff={"r": 4096, "w": 1936}, lru_width=1280, blocks=5, taps=4, wkv_heads=17, wkv_dim=64, wkv_rank=96),
    "plain": synthetic.looped_shape("pgp", width=2048, vocab=336, ff={"p": 4040, "g": 2856}, loop=(1, 2, 2), heads=4, kv_heads=2, delta_heads=4, delta_kv_heads=2,
                                    delta_rank=144, gate_rank=72, gla_heads=11, gla_rank=80),
}
#: rows so long that few of them are cut in four along K, with tiles of 64 tokens of either width (fp32: its tokens' side in parts)
LONG = synthetic.hybrid_shape("a", width=2048, vocab=336, streams=2, ff={"a": 8192}, heads=2, dim=128, rot_dim=64, v_dim=128, rank=128, window=512)
LONG_LENGTHS = (200, 260)


@functools.lru_cache(maxsize=None)
def expected(name):
    shape = {**SHAPES, "long": LONG}[name]
    w = synthetic.random_hybrid_weights(shape, 3, DEVICE)
    tokens = torch.randint(0, shape.vocab, (MOST,), generator=torch.Generator().manual_seed(5))
    with torch.device(DEVICE):
        oracle = givopel_oracle if shape.plain else O
        return w, tokens, oracle.forward(shape.to_config(), w, tokens.to(DEVICE), dtype=torch.float64)     # causal: a prefix's logits are its rows


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_products_at_the_edges_of_tiles(name, n, dtype):
    check(name, SHAPES[name], n, dtype)


@pytest.mark.parametrize("n", LONG_LENGTHS)
def test_long_rows_cut_in_four(n):
    check("long", LONG, n, torch.float32)


def check(name, shape, n, dtype):
    w, tokens, want = expected(name)
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=MOST, portion_rows=MOST)
    got = decode_hybrid.run_tokens(g, mk_kernel.get_mk(), RequestTable(g).open(0), tokens[:n], range(n)).double()
    d = got - want[:n]
    d = d - d.mean(-1, keepdim=True)
    err = float((d.pow(2).mean(-1).sqrt() / want[:n].pow(2).mean().sqrt()).max())
    assert err < (TOL_PLAIN if shape.plain else TOL)[dtype], f"{err:.3g}"


@pytest.mark.parametrize("width,channels", [(208, 160), (256, 192)], ids=["whole", "parts"])
def test_values_that_are_not_finite_stay_so_in_fp32(width, channels):
    """An infinite or undefined embedding reaches the logits of its token as such, and none of a token before it.  (A
    recurrence: an attention's weight of zero times an undefined value is undefined.)"""
    shape = synthetic.hybrid_shape("r", width=width, vocab=96, streams=2, ff={"r": channels + 16 * (width == 208)}, lru_width=channels, blocks=1, taps=3)
    w = synthetic.random_hybrid_weights(shape, 6, DEVICE)
    w["embed"][7, 3] = float("inf")
    w["embed"][8, 5] = float("nan")
    ids = torch.arange(40) % 6
    ids[20], ids[30] = 7, 8
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=torch.float32, max_positions=64, portion_rows=64)
    got = decode_hybrid.run_tokens(g, mk_kernel.get_mk(), RequestTable(g).open(0), ids, range(40))
    assert torch.isfinite(got[:20]).all()
    assert not torch.isfinite(got[20]).any() and not torch.isfinite(got[30]).any()


@pytest.mark.parametrize("width", [208, 256, 704], ids=["whole", "parts", "parts, cut"])
def test_infinite_weights_in_fp32(width):
    """A finite value times an infinite weight is infinite, also where some of the value's three parts are zero."""
    shape = synthetic.hybrid_shape("r", width=width, vocab=160, streams=2, lru_width=96, blocks=1, taps=3)
    w = synthetic.random_hybrid_weights(shape, 6)
    for i in range(shape.vocab):
        w["head"][i, i] = float("inf") if i % 3 else -float("inf")
    ids = torch.randint(0, shape.vocab, (130,), generator=torch.Generator().manual_seed(2))
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=torch.float32, max_positions=160, portion_rows=160)
    got = decode_hybrid.run_tokens(g, mk_kernel.get_mk(), RequestTable(g).open(0), ids, range(130)).cpu()
    want = O.forward(shape.to_config(), w, ids, dtype=torch.float64)
    assert torch.isinf(want).all() and torch.equal(got.double(), want)


@pytest.mark.parametrize("byte", [0x01, 0xFF], ids=["ones", "undefined values"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("shape", [SHAPES["large"], synthetic.looped_shape("pg", width=2048, vocab=96, ff={"p": 2048}, heads=2, kv_heads=1, delta_heads=2,
                                                                          delta_kv_heads=1, gla_heads=2)], ids=["streams", "plain"])
def test_a_workspace_that_has_held_something_else(shape, dtype, byte):
    """Decode and prefill launches may share a buffer: nothing a launch finds in it counts."""
    g = build_globals(shape, weights.pack(shape, synthetic.random_hybrid_weights(shape, 4, DEVICE), DEVICE), dtype=dtype, max_positions=64, portion_rows=64)
    mk, tokens, got = mk_kernel.get_mk(), torch.arange(40) % shape.vocab, []
    for fill in (0, byte):
        table = RequestTable(g)
        request, parts = table.open(0), []
        for part in tokens.split([20, 1, 18, 1]):
            if got:
                mk._prefill_ws.fill_(fill)
                mk._decode_ws.fill_(fill)
            parts.append(decode_hybrid.run_tokens(g, mk, request, part, range(len(part))))
        mk.check()
        got.append(torch.cat(parts))
    assert torch.isfinite(got[0]).all() and torch.equal(got[0], got[1])
