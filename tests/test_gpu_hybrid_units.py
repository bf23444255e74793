"""The decode kernel's tagged units: vectors around what a workgroup's threads hold and look at together, and a workspace that keeps nothing."""
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
TAGS = range(0x5E000000, 0x5E100000)      # kTagBase, kTags


def streams(width, ff):
    return synthetic.hybrid_shape("raw", width=width, vocab=96, streams=2, ff={"r": ff, "a": 64}, heads=18, dim=32, rot_dim=96, v_dim=32, rank=496, window=40, lru_width=96, blocks=2,
                                  taps=5, wkv_heads=2, wkv_dim=64, wkv_rank=24)


def plain(width, ff):
    return synthetic.looped_shape("pgg", width=width, vocab=96, ff={"p": ff, "g": 32}, loop=(1, 2, 2), heads=40, kv_heads=2, dim=64, v_dim=32, delta_heads=10, delta_kv_heads=5,
                                  delta_dim=48, delta_v_dim=80, delta_rank=24, gate_rank=40, gla_heads=9, gla_dim=32, gla_v_dim=208, gla_rank=16)


def on_gpu(shape, dtype):
    w = synthetic.random_hybrid_weights(shape, 3)
    return w, build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=64)


def tags_left(mk):
    words = mk._decode_ws.view(torch.int32)
    return int(((words >= TAGS.start) & (words < TAGS.stop)).sum())


# Widths below, at and behind 2048 values (four a thread) and twice that; feed-forwards around 2048 + 12 x 512.  Queries of eighteen and twenty heads a group take two
# instructions, of 496 + 96 columns two rounds of looks.
@pytest.mark.parametrize("dtype, tolerance", [(torch.float32, 4e-5), (torch.bfloat16, 8e-2)], ids=["fp32", "bf16"])      # as in the routes' own tests
@pytest.mark.parametrize("width, ff", [(2032, 8192), (2048, 8208), (2064, 2048), (4112, 14352)])
@pytest.mark.parametrize("kind", [streams, plain])
def test_steps(kind, width, ff, dtype, tolerance):
    shape = kind(width, ff)
    w, g = on_gpu(shape, dtype)
    mk, ids = mk_kernel.get_mk(), torch.arange(5, 11)
    request = RequestTable(g).open(0)
    got = torch.cat([decode_hybrid.run_tokens(g, mk, request, ids[i : i + 1], [0]) for i in range(len(ids))]).double().cpu()
    mk.check()
    oracle = hybrid_oracle if kind is streams else givopel_oracle
    want = oracle.forward(shape.to_config(), w, ids, dtype=torch.float64)
    d = got - want
    d = d - d.mean(-1, keepdim=True)
    assert float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max()) < tolerance
    assert tags_left(mk) == 0


@pytest.mark.parametrize("kind", [streams, plain])
def test_a_failed_step_leaves_no_unit(kind):
    shape = kind(2048, 2048)
    _, g = on_gpu(shape, torch.bfloat16)
    table, steps = RequestTable(g), []
    for limit in (0, 1, 0):
        mk = mk_kernel.get_mk(spin_limit=limit) if limit else mk_kernel.get_mk()
        request, out = table.open(0), []
        for token in range(3):
            out.append(decode_hybrid.run_tokens(g, mk, request, [token], [0]).clone())
        if limit:
            with pytest.raises(RuntimeError, match="ran out of polls"):
                mk.check()
        else:
            mk.check()
            steps.append(torch.cat(out))
        assert tags_left(mk) == 0 and int(g.barriers.abs().sum()) == 0
        table.close(0)
    assert torch.equal(*steps)
