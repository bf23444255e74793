"""Recurrences of portions walked in segments: portions that end at, one ahead of and one behind a chunk, a segment, the most segments that put their own starts
together (four of 128 tokens) and the most chunks that fp32 walks in one go (sixteen); heads of every number of tiles a wave takes, values off the 64 columns of a
workgroup.  A second portion and a token start from the state that the first one leaves."""
import functools

import pytest
import torch

import givopel_oracle
import hybrid_oracle
from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu

DEVICE = "cuda:0"
MOST = 660
SHAPES = {
    "wkv 16": synthetic.hybrid_shape("w", width=64, vocab=96, streams=2, wkv_heads=5, wkv_dim=16, wkv_rank=16),
    "wkv 80": synthetic.hybrid_shape("w", width=80, vocab=96, streams=1, wkv_heads=3, wkv_dim=80, wkv_rank=16),
    "wkv 250": synthetic.hybrid_shape("w", width=64, vocab=96, streams=2, wkv_heads=2, wkv_dim=250, wkv_rank=20),
    "gla 64 | 80": synthetic.looped_shape("g", width=64, vocab=96, gla_heads=3, gla_dim=64, gla_v_dim=80, gla_rank=16),
    "gla 120 | 48": synthetic.looped_shape("g", width=96, vocab=96, gla_heads=2, gla_dim=120, gla_v_dim=48, gla_rank=16, tau=2.0),
    "gla 256 | 130": synthetic.looped_shape("g", width=64, vocab=96, gla_heads=2, gla_dim=256, gla_v_dim=130, gla_rank=12),
    "delta 48 | 112": synthetic.looped_shape("p", width=64, vocab=96, heads=2, kv_heads=1, dim=16, v_dim=16, delta_heads=4, delta_kv_heads=2, delta_dim=48, delta_v_dim=112,
                                             taps=3, delta_rank=16, gate_rank=16),
}
#: as in the routes' own tests
TOLERANCE = {(hybrid_oracle, torch.float32): 2e-5, (hybrid_oracle, torch.bfloat16): 4e-2, (givopel_oracle, torch.float32): 4e-5, (givopel_oracle, torch.bfloat16): 8e-2}


@functools.lru_cache(maxsize=None)
def model(name):
    shape, oracle = SHAPES[name], hybrid_oracle if name.startswith("wkv") else givopel_oracle
    w, ids = synthetic.random_hybrid_weights(shape, 2), torch.randint(0, shape.vocab, (MOST,), generator=torch.Generator().manual_seed(8))
    return shape, oracle, w, ids, oracle.forward(shape.to_config(), w, ids, dtype=torch.float64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("name", SHAPES)
def test_portions(name, dtype):
    shape, oracle, w, ids, want = model(name)
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=MOST, portion_rows=640)
    mk, table = mk_kernel.get_mk(), RequestTable(g)
    for n in (15, 16, 17, 127, 128, 129, 255, 256, 257, 511, 512, 513, 640):
        request, got, at = table.open(n), [], 0
        for part in (n, 1, 18):
            got.append(decode_hybrid.run_tokens(g, mk, request, ids[at : at + part], range(part)))
            at += part
        mk.check()
        table.close(n)
        d = torch.cat(got).double().cpu() - want[:at]
        d = d - d.mean(-1, keepdim=True)
        err = float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max())
        assert err < TOLERANCE[oracle, dtype], f"{n} tokens: {err:.3g}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("n, at", [(40, 20), (40, 39), (330, 261)], ids=["inside a chunk", "the last token", "a later segment"])
@pytest.mark.parametrize("what", ["gla, undefined embedding", "wkv, undefined embedding", "wkv, infinite embedding", "wkv, infinite keys", "wkv, infinite values"])
def test_a_token_that_is_not_finite_reaches_none_before_it(what, n, at, dtype):
    kind, what = what.split(", ")
    shape = SHAPES["wkv 80" if kind == "wkv" else "gla 64 | 80"]
    w = synthetic.random_hybrid_weights(shape, 5)
    if what.endswith("embedding"):
        w["embed"][7, 3] = float("nan" if what.startswith("undefined") else "inf")
    else:       # a column of the weights that this token alone meets
        w["embed"][:, 3] = 0
        w["embed"][7] = 0
        w["embed"][7, 3] = 1
        w["l0.mix." + what.split()[1][0]][:, 3] = 3e38
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=MOST, portion_rows=640)
    mk, ids, got = mk_kernel.get_mk(), torch.arange(n) % 6, []
    for token in (5, 7):
        ids[at] = token
        table = RequestTable(g)
        got.append(decode_hybrid.run_tokens(g, mk, table.open(0), ids, range(n)))
        table.close(0)
    mk.check()
    assert torch.isfinite(got[0]).all() and torch.equal(got[0][:at], got[1][:at])
    assert not torch.isfinite(got[1][at:]).any(dim=-1).any()


@pytest.mark.parametrize("n", [250, 640])
def test_states_that_do_not_fade_are_summed_by_chunks(n):
    """A state of n tokens without decay.  A sum by tokens is rounded n times, each time by up to half a last place (2^-24 / sqrt 3 evenly spread, three quarters of it on the average
    place between two powers of two: 2.6e-8) of the sum so far: sqrt(n / 2) x 2.6e-8 of the last one.  A sum by chunks of sixteen tokens is rounded a sixteenth as often, so a quarter as
    far; keys and values bring up to 1e-7."""
    shape = synthetic.hybrid_shape("w", width=128, vocab=96, streams=1, wkv_heads=2, wkv_dim=64, wkv_rank=16)
    w, ids = synthetic.random_hybrid_weights(shape, 2), torch.randint(0, 96, (n,), generator=torch.Generator().manual_seed(8))
    w["l0.mix.w2"].zero_()
    w["l0.mix.w0"].fill_(-30)      # decays of one, to 1e-13
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=torch.float32, max_positions=MOST, portion_rows=640)
    mk, request = mk_kernel.get_mk(), RequestTable(g).open(0)
    decode_hybrid.run_tokens(g, mk, request, ids)
    mk.check()
    d = {name: t.double() for name, t in w.items()}
    x = d["embed"][ids] * d["l0.hc1.in"]
    h = x / torch.sqrt((x * x).mean(-1, keepdim=True) + shape.eps) * d["l0.norm1"]
    before = torch.cat((torch.zeros_like(h[:1]), h[:-1]))
    k, v = (((h + (before - h) * d["l0.mix.mu." + c]) @ d["l0.mix." + c].T).view(n, 2, 64) for c in "kv")
    want = torch.stack([k[:, head].T @ v[:, head] for head in range(2)])
    got = g.layer_state[0]["state"][0].double().cpu().view_as(want)
    err = float((got - want).norm() / want.norm())
    assert err < 1e-7 + 0.25 * (n / 2) ** 0.5 * 2.6e-8, f"{err:.3g}"
