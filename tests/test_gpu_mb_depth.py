"""The tiles engine's attention with four tiles of keys a wave in flight (up to three slices a head) against two (four slices), and its schedules of 5 to 16 rows.

Contexts around the tiles that a wave holds (8 waves x 16 tokens x 4) and their refills, a slice that ends inside a tile, and one without keys.  The
slices' sums are the same fp32 products added in another order, over at most 1300 keys, and rounded to bf16 once: at most one step apart.
"""
import dataclasses

import pytest
import torch

from fused_mb_oracle import FusedBatchOracle
from gpu_helpers import bf16_close, rel_close, tensor_rel_close
from qimeng_megakernel_amd import synthetic
from qimeng_megakernel_amd.decode_schedule.model_config import LLAMA_3_2_1B, QWEN3_1_7B, LlamaConfig
from qimeng_megakernel_amd.decode_schedule_mb import mk_kernel
from qimeng_megakernel_amd.decode_schedule_mb.instructions import scheduler as S
from qimeng_megakernel_amd.decode_schedule_mb.row_state import RowState

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


# Rows and capacities on both sides of the schedule's lines: one slice, or two or three beside the QKV blocks or behind them; counter rows widened for 5 to 7 rows.
STEPS = [(QWEN3_1_7B, 5, 640, 1), (QWEN3_1_7B, 5, 656, 3), (QWEN3_1_7B, 5, 6016, 4), (QWEN3_1_7B, 6, 656, 2), (QWEN3_1_7B, 7, 1040, 4), (QWEN3_1_7B, 9, 1024, 1), (QWEN3_1_7B, 9, 1040, 3),
         (QWEN3_1_7B, 12, 1040, 2), (QWEN3_1_7B, 16, 1024, 1), (QWEN3_1_7B, 16, 1040, 2), (LLAMA_3_2_1B, 5, 1024, 1), (LLAMA_3_2_1B, 5, 1040, 4), (LLAMA_3_2_1B, 6, 2064, 3)]


@pytest.mark.parametrize("full,rows,capacity,slices", STEPS, ids=lambda v: f"heads_of_{v.head_dim}" if hasattr(v, "head_dim") else str(v))
def test_steps_of_the_template(full, rows, capacity, slices):
    """Two whole steps of two full-width layers against the fused oracle, from the schedule of that many rows and positions: hidden states and logits within the gates
    of the other whole steps, counters cleared behind each."""
    shape = dataclasses.replace(full, num_hidden_layers=2, vocab_size=512)
    LlamaConfig.set_shape(shape)
    sched = S.mi355x_scheduler(rows, shape)
    assert sched.partials_for_capacity(capacity) == slices
    weights = synthetic.random_weights(shape, 3, max_positions=capacity)
    cpu, gpu = (synthetic.build_batch_globals(weights, shape, capacity, rows, device) for device in ("cpu", "cuda:0"))
    gen = torch.Generator().manual_seed(rows)
    last = min(capacity, 1100) - 2
    start = torch.tensor([last - last * r // rows for r in range(rows)], dtype=torch.int32)       # ragged; at the end of the cache where it is short
    for name in ("k_cache", "v_cache"):
        filled = torch.randn(2, rows, last, shape.num_key_value_heads, shape.head_dim, generator=gen).bfloat16()
        getattr(cpu, name)[:, :, :last].copy_(filled)
        getattr(gpu, name)[:, :, :last].copy_(filled)
    for g in (cpu, gpu):
        g.position_ids.copy_(start)
        RowState.of(g)
    assert gpu.barriers.shape[2] >= mk_kernel.BatchMegaKernel.XCD_COUNTER_WORDS
    mk_kernel.build(gpu)
    mk, oracle = mk_kernel.get_mk(spin_limit=1 << 18), FusedBatchOracle(shape)
    for step in range(2):
        print(f"{rows} rows of {capacity}, step {step}", flush=True)
        hidden = (torch.randn(rows, shape.hidden_size, generator=gen) * 0.7).bfloat16()
        for g in (cpu, gpu):
            g.hidden_states.copy_(hidden)
            g.position_ids.copy_(start + step)
        oracle.decode_step(cpu)
        mk_kernel.call_mk(gpu, mk)
        mk.check()
        tensor_rel_close(gpu.hidden_states, cpu.hidden_states, name="hidden_states")
        rel_close(gpu.logits, cpu.logits, rel=4e-2, name="logits")
        assert int(gpu.barriers.abs().sum()) == 0
