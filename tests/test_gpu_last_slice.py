"""Tagged launches with many split-KV slices, where the slice that arrives last on a KV head merges its group, against launches on
counters, where every O-projection workgroup merges all heads: the same operations in the same order, so the same bits.

Fan-outs around the line between the two (4 | 5), around the sixteen slices of a trip, the widest, and a cache that leaves slices
empty."""
import dataclasses

import pytest
import torch

from qimeng_megakernel_amd import synthetic
from qimeng_megakernel_amd.decode_schedule import mk_kernel
from qimeng_megakernel_amd.decode_schedule.instructions import scheduler as S
from qimeng_megakernel_amd.decode_schedule.model_config import LLAMA_3_2_1B, QWEN3_1_7B, LlamaConfig

pytestmark = pytest.mark.gpu

CAPACITY = 1100
BUFFERS = ("hidden_states", "q_post_rope", "attn_out", "silu_out", "logits", "k_cache", "v_cache", "attn_out_intermediates", "attn_lse_intermediates")


@pytest.mark.parametrize("xcd", [True, False], ids=["sub-counters", "counter rows"])
@pytest.mark.parametrize("slices,position", [(4, 1000), (5, 1000), (15, 1077), (16, 640), (17, 1000), (32, 1099), (32, 40)])
@pytest.mark.parametrize("model", ["llama", "qwen"])
def test_last_slice_merges_to_the_same_bits(model, slices, position, xcd):
    shape = dataclasses.replace(LLAMA_3_2_1B if model == "llama" else QWEN3_1_7B, num_hidden_layers=2, vocab_size=512)
    LlamaConfig.set_shape(shape)
    w = synthetic.random_weights(shape, 5, CAPACITY)
    gen = torch.Generator().manual_seed(slices)
    past = [torch.randn(2, 1, CAPACITY, shape.num_key_value_heads, shape.head_dim, generator=gen).bfloat16() for _ in range(2)]
    done = []
    for tagged in (False, True):
        g = synthetic.build_globals(w, shape, CAPACITY, "cuda:0")
        g.k_cache.copy_(past[0])
        g.v_cache.copy_(past[1])
        mk = mk_kernel.get_mk(tagged=tagged, xcd_counters=xcd)
        S.tensorize_instructions(g, S.mi355x_scheduler(shape, num_partials=slices).queues())
        for step in range(3):      # the counters are back where they were after every launch
            g.hidden_states.copy_(g.embed_tokens[11 + step])
            g.position_id = position - step
            mk_kernel.call_mk(g, mk)
        mk.check()
        assert mk._tagged == tagged and not int(g.barriers.abs().sum())
        done.append(g)
    for name in BUFFERS:
        assert torch.equal(getattr(done[0], name), getattr(done[1], name)), name


def test_a_fan_out_beyond_the_workspace_is_rejected():
    """As where the O-projection reads the partials itself: an operand error, not a wait that runs out."""
    shape = dataclasses.replace(LLAMA_3_2_1B, num_hidden_layers=1, vocab_size=512)
    LlamaConfig.set_shape(shape)
    g = synthetic.build_globals(synthetic.random_weights(shape, 5, 64), shape, 64, "cuda:0")
    mk = mk_kernel.get_mk(tagged=True, spin_limit=20000)
    S.tensorize_instructions(g, S.mi355x_scheduler(shape, num_partials=8).queues())
    oproj = g.instructions[:, :, 0] == 4
    assert set(g.instructions[..., 5][oproj].tolist()) == {8} and (splits := g.attn_lse_intermediates.shape[1]) < 64
    g.instructions[..., 5][oproj] = splits + 1
    g.position_id = 40
    mk_kernel.call_mk(g, mk)
    assert mk._tagged
    with pytest.raises(RuntimeError, match="operand out of bounds") as err:
        mk.check()
    assert "opcode=4" in str(err.value) and "operand=5" in str(err.value)
