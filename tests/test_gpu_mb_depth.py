"""The tiles engine's attention with four tiles of keys a wave in flight (up to three slices a head) against two (four slices).

Contexts around the tiles that a wave holds (8 waves x 16 tokens x 4) and their refills, a slice that ends inside a tile, and one without keys.  The
slices' sums are the same fp32 products added in another order, over at most 1300 keys, and rounded to bf16 once: at most one step apart.
"""
import dataclasses

import pytest
import torch

from gpu_helpers import bf16_close
from qimeng_megakernel_amd import synthetic
from qimeng_megakernel_amd.decode_schedule.model_config import LLAMA_3_2_1B, QWEN3_1_7B, LlamaConfig
from qimeng_megakernel_amd.decode_schedule_mb import mk_kernel
from qimeng_megakernel_amd.decode_schedule_mb.instructions import scheduler as S

pytestmark = pytest.mark.gpu

POSITIONS = (0, 15, 510, 511, 512, 640, 1023, 1299)


@pytest.mark.parametrize("full", [LLAMA_3_2_1B, QWEN3_1_7B], ids=lambda s: f"heads_of_{s.head_dim}")
@pytest.mark.parametrize("slices", [1, 2, 3])
def test_tiles_ahead(full, slices, monkeypatch):
    print(f"heads of {full.head_dim}, {slices} slices", flush=True)
    shape, rows, capacity = dataclasses.replace(full, num_hidden_layers=1, vocab_size=512), len(POSITIONS), 1300
    LlamaConfig.set_shape(shape)
    weights = synthetic.random_weights(shape, 3, max_positions=capacity)
    gen = torch.Generator().manual_seed(slices)
    hidden = (torch.randn(rows, shape.hidden_size, generator=gen) * 0.7).bfloat16()
    past = [torch.randn(1, rows, capacity, shape.num_key_value_heads, shape.head_dim, generator=gen).bfloat16() for _ in range(2)]
    out = []
    for p in (4, slices):
        monkeypatch.setattr(S.BatchScheduler, "_fan_out", lambda self, r, b, p=p: p)
        g = synthetic.build_batch_globals(weights, shape, capacity, rows, "cuda:0")
        g.hidden_states.copy_(hidden)
        g.k_cache.copy_(past[0])
        g.v_cache.copy_(past[1])
        g.position_ids.copy_(torch.tensor(POSITIONS, dtype=torch.int32))
        mk_kernel.build(g)
        mk = mk_kernel.get_mk(spin_limit=1 << 18)
        mk_kernel.call_mk(g, mk)
        mk.check()
        out.append(g.attn_out.cpu())
    bf16_close(out[1], out[0], ulps=1.0, name="attn_out")


def test_both_kernels_of_heads_of_64():
    """Caches of 2048 and 2064 positions take the kernels of four and of two tiles ahead: the same tiles in the same order, the same bits."""
    shape, rows, out = dataclasses.replace(LLAMA_3_2_1B, num_hidden_layers=1, vocab_size=512), len(POSITIONS), []
    LlamaConfig.set_shape(shape)
    weights = synthetic.random_weights(shape, 3, max_positions=2064)
    gen = torch.Generator().manual_seed(9)
    hidden = (torch.randn(rows, shape.hidden_size, generator=gen) * 0.7).bfloat16()
    past = [torch.randn(1, rows, 2048, shape.num_key_value_heads, shape.head_dim, generator=gen).bfloat16() for _ in range(2)]
    for capacity in (2048, 2064):
        print(f"capacity {capacity}", flush=True)
        g = synthetic.build_batch_globals(weights, shape, capacity, rows, "cuda:0")
        g.hidden_states.copy_(hidden)
        g.k_cache[:, :, :2048].copy_(past[0])
        g.v_cache[:, :, :2048].copy_(past[1])
        g.position_ids.copy_(torch.tensor([*POSITIONS[:-1], 2047], dtype=torch.int32))
        mk_kernel.build(g, 2048)                      # one slice in either
        mk = mk_kernel.get_mk(spin_limit=1 << 18)
        mk_kernel.call_mk(g, mk)
        mk.check()
        out.append((g.attn_out.cpu(), g.hidden_states.cpu(), g.logits.cpu()))
    assert all(torch.equal(a, b) for a, b in zip(*out))
