"""The prefill's bf16 attention (csrc/qmk_hybrid_attention.h) at the edges of its tiles: 64 queries a workgroup, 16 a wave, stages of 64 or 32 keys,
windows and pasts that start and end inside them, heads of every size it is compiled for; against the plain implementation in 64 bits, bf16's tolerances as in
test_gpu_hybrid.py and, on a plain residual, test_gpu_looped.py.  The workspace holds what is no number before each portion.

Queries are drawn twice as large and output projections eight times, so that single keys count: test_attention_faults.py holds that one key more or less at a window's
end, or one missing in every 32, is far outside the tolerance on every shape."""
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
MOST = 330


def latent(**sizes):
    return synthetic.hybrid_shape("a", vocab=96, streams=2, **{"width": 128, "rank": 64, **sizes})


SHAPES = {
    "96 | 48, window 40": latent(heads=3, dim=64, rot_dim=32, v_dim=48, window=40),
    "112 | 112, window 77": latent(heads=3, dim=80, rot_dim=32, v_dim=112, window=77),
    "192 | 128, window 101": latent(heads=9, dim=128, rot_dim=64, v_dim=128, window=101),
    "256 | 208, window 129": latent(heads=2, dim=200, rot_dim=40, v_dim=200, window=129),
    "grouped 128 | 128": synthetic.looped_shape("p", width=256, vocab=96, heads=8, kv_heads=2, delta_heads=2, delta_kv_heads=2, delta_dim=32, delta_v_dim=32, delta_rank=16, gate_rank=16),
}


def tolerance(shape):
    return 8e-2 if shape.plain else 4e-2


def inputs(name):
    """Shape, weights and tokens, the same on every machine."""
    shape = SHAPES[name]
    w = synthetic.random_hybrid_weights(shape, 3)
    for part, times in ((".mix.q", 2), (".mix.left.q", 2), (".mix.o", 8), (".mix.left.o", 8)):
        w.update({key: t * times for key, t in w.items() if key.endswith(part)})
    return shape, w, torch.randint(0, shape.vocab, (MOST,), generator=torch.Generator().manual_seed(5))


def worst(got, want):
    """Largest error of a token's logits, as a root mean square over theirs."""
    d = got.double() - want
    d = d - d.mean(-1, keepdim=True)
    return float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max())


@functools.lru_cache(maxsize=None)
def model(name):
    shape, w, tokens = inputs(name)
    w = {key: t.to(DEVICE) for key, t in w.items()}
    with torch.device(DEVICE):
        want = (givopel_oracle if shape.plain else hybrid_oracle).forward(shape.to_config(), w, tokens.to(DEVICE), dtype=torch.float64)
    return shape, w, tokens, want


@pytest.mark.parametrize("past,n", [(0, 2), (0, 31), (0, 33), (0, 64), (0, 65), (0, 200), (1, 63), (31, 16), (32, 33), (45, 130), (64, 64), (200, 2), (199, 129)])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_attention_at_the_edges_of_its_tiles(name, past, n):
    shape, w, tokens, want = model(name)
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=torch.bfloat16, max_positions=MOST, portion_rows=MOST)
    mk, request = mk_kernel.get_mk(), RequestTable(g).open(0)
    got = []
    for start, end in ((0, past), (past, past + n)):
        if end == start:
            continue
        mk._bind(g)
        mk._prefill_ws.fill_(0xFF)
        got.append(decode_hybrid.run_tokens(g, mk, request, tokens[start:end], range(end - start)))
    err = worst(torch.cat(got), want[: past + n])
    assert err < tolerance(shape), f"{err:.3g}"


@pytest.mark.parametrize("name", sorted(n for n, shape in SHAPES.items() if not shape.plain))
@pytest.mark.parametrize("at", [3, 40, 100])
def test_an_undefined_value_stays_out_of_what_no_query_of_a_wave_sees(name, at):
    """Sixteen queries take 32 keys together, with weights of zero where one does not see a key; keys that none of the sixteen sees do not enter at all."""
    shape, w, tokens, _ = model(name)
    n, window, undefined = 200, shape.entries[0].shape.window, shape.vocab - 1
    tokens = tokens[:n].clamp(max=undefined - 1).index_fill(0, torch.tensor([at]), undefined)
    w = {**w, "embed": w["embed"].index_fill(0, torch.tensor([undefined], device=DEVICE), float("nan"))}
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=torch.bfloat16, max_positions=n, portion_rows=n)
    got = decode_hybrid.run_tokens(g, mk_kernel.get_mk(), RequestTable(g).open(0), tokens, range(n))
    defined, block = torch.isfinite(got).all(-1).tolist(), at & ~31
    for i in range(n):
        wave = i & ~15
        if block > wave + 15 or wave - (block + 31) >= window:      # none of its sixteen queries sees any of the 32 keys
            assert defined[i], i
        if 0 <= i - at < window:
            assert not defined[i], i
