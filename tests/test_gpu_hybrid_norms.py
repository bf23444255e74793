"""bf16 portions take a norm's factor behind the product, from sums of squares that the product before leaves: at the edges of a run of 128 columns, of the tiles
that leave and read them, and on both sides of the largest width, against the plain implementation and with a token's bits the same in every length."""
import pytest
import torch

import hybrid_oracle as O
from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [64, 192, 1088, 2048, 2112])
def test_factors_of_tokens(width):
    shape = synthetic.hybrid_shape("aa", width=width, vocab=96, streams=2, ff={"a": 448}, heads=2, dim=32, rot_dim=16, v_dim=32, rank=64, window=500)
    w = synthetic.random_hybrid_weights(shape, 3)
    w["embed"] *= torch.logspace(-3, 1, 96)[:, None].to(w["embed"].dtype)      # tokens of very different size: a factor that is another token's shows
    most = 700
    ids = torch.randint(0, shape.vocab, (most,), generator=torch.Generator().manual_seed(1))
    want = O.forward(shape.to_config(), w, ids[:140], dtype=torch.float64)
    g = build_globals(shape, weights.pack(shape, w, "cuda:0"), dtype=torch.bfloat16, max_positions=most + 8, portion_rows=most)
    mk, table = mk_kernel.get_mk(), RequestTable(g)

    def logits(n):
        got = decode_hybrid.run_tokens(g, mk, table.open(n), ids[:n], range(n))
        table.close(n)
        mk.check()
        return got

    whole = logits(most)
    d = whole[:140].double().cpu() - want
    d = d - d.mean(-1, keepdim=True)
    # bf16 keeps eight bits: 2 layers of some ten roundings each, of 2^-9 of their values, add up to 2^-9 sqrt(20) = 0.009 of the logits on the average; a single token's are some times that.
    assert float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max()) < 8e-2
    for n in (2, 31, 64, 65, 97, 140, 257, 520):
        assert torch.equal(logits(n), whole[:n]), n
