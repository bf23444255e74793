"""The prefill's bf16 attention with 64 queries a workgroup and with 16 whose waves share a stage's work (csrc/qmk_hybrid_attention.h): the bits of a token's logits
do not depend on which of them its portion's length takes.  Twenty heads of 192 take 64 from 193 tokens on in
bf16 and fp32, forty of 128 from 193 and from 97.  (The shorter portions are held to
64 bits by test_gpu_hybrid_attention.py.)"""
import functools

import pytest
import torch

from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu

DEVICE = "cuda:0"
MOST = 440
SHAPES = {
    "192 | 128, window 101": synthetic.hybrid_shape("a", vocab=96, streams=2, width=128, rank=64, heads=20, dim=128, rot_dim=64, v_dim=128, window=101),
    "160 | 80": synthetic.hybrid_shape("a", vocab=96, streams=2, width=128, rank=64, heads=20, dim=128, rot_dim=32, v_dim=80, window=500),
    "grouped 128 | 128": synthetic.looped_shape("p", width=256, vocab=96, heads=40, kv_heads=4, delta_heads=2, delta_kv_heads=2, delta_dim=32, delta_v_dim=32, delta_rank=16, gate_rank=16),
}


@functools.lru_cache(maxsize=None)
def model(name, dtype=torch.bfloat16):
    shape = SHAPES[name]
    w = {key: t.to(DEVICE) * (8 if key.endswith((".mix.o", ".mix.left.o")) else 1) for key, t in synthetic.random_hybrid_weights(shape, 3).items()}
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=MOST, portion_rows=MOST)
    return g, torch.randint(0, shape.vocab, (MOST,), generator=torch.Generator().manual_seed(5))


def logits(g, tokens, past, count):
    table = RequestTable(g)
    request, mk = table.open(0), mk_kernel.get_mk()
    if past:
        decode_hybrid.run_tokens(g, mk, request, tokens[:past])
    got = decode_hybrid.run_tokens(g, mk, request, tokens[past : past + count], range(count))
    table.close(0)
    return got


@pytest.mark.parametrize("past,n", [(0, 209), (0, 256), (31, 240), (64, 257), (199, 211)])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_few_queries_come_out_as_many_do(name, past, n):
    g, tokens = model(name)
    many = logits(g, tokens, past, n)
    assert torch.isfinite(many).all()
    for count in (2, 37, 64, 192):
        assert torch.equal(logits(g, tokens, past, count), many[:count]), count


@pytest.mark.parametrize("past,n", [(0, 209), (31, 240), (199, 211)])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_few_queries_in_float32(name, past, n):
    """Keys go to four waves' sums instead of two groups': the order differs, and with it the last bits (2^-24 each of a few hundred additions)."""
    g, tokens = model(name, torch.float32)
    many, few = logits(g, tokens, past, n), logits(g, tokens, past, 96)
    d = (many[:96].double() - few.double()).pow(2).mean(-1).sqrt() / many.double().pow(2).mean().sqrt()
    assert float(d.max()) < 256 * 2.0**-24, float(d.max())
