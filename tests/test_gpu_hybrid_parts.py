"""The parts of a decode step's attention, also those without a key: they wait like the others, since what they leave takes the place of parts that the attention
before may still be merging (test_hybrid_handover.py works out where)."""
import pytest
import torch

import givopel_oracle
import hybrid_oracle
from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.instructions import instruction_defs as D
from qimeng_megakernel_amd.decode_schedule_hybrid.instructions.scheduler import tensorize
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable
from test_hybrid_handover import SMALL, uneven, uneven_plain

pytestmark = pytest.mark.gpu

DEVICE = "cuda:0"
BOTH = pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])


@BOTH
@pytest.mark.parametrize("shape", [uneven(64, [SMALL]), uneven_plain(64, [{}])], ids=["streams", "plain"])
def test_a_part_without_keys_waits_for_its_layer(shape, dtype):
    """Alone in a launch nothing makes its queries: its looks run out."""
    g = build_globals(shape, weights.pack(shape, synthetic.random_hybrid_weights(shape, 2), DEVICE), dtype=dtype, max_positions=256)
    RequestTable(g).open(0)
    mk = mk_kernel.get_mk(spin_limit=50)
    part = D.AttendSplitKV(0, 0, 1, 2)
    g.instructions, g.instruction_splits = tensorize([[part]], DEVICE), 2
    g.barriers = torch.zeros(1, 54, 48, dtype=torch.int32, device=DEVICE)
    mk(g)      # position 0: all keys there are belong to part 0
    with pytest.raises(RuntimeError, match="ran out of polls") as err:
        mk.check()
    assert "opcode=4" in str(err.value)


#: fewer output blocks than queues; parts without keys beside parts that have some, at the same places or not
SHAPES = {
    "windows": uneven(64, [dict(SMALL, window=190), dict(SMALL, window=70), dict(SMALL, window=190)]),
    "ranks": uneven(64, [dict(SMALL, rank=272), dict(SMALL, rank=144), dict(SMALL, rank=16, heads=2)]),
    "heads": uneven(48, [dict(heads=18, rank=144), dict(heads=2, rank=400, window=40), dict(heads=33, rank=64)]),
    "plain": uneven_plain(64, [dict(heads=2), dict(heads=40, v_dim=80), dict(heads=4, kv_heads=4, v_dim=200)]),
}
#: as in the routes' own tests
TOLERANCE = {(False, torch.float32): 2e-5, (False, torch.bfloat16): 4e-2, (True, torch.float32): 4e-5, (True, torch.bfloat16): 8e-2}


@BOTH
@pytest.mark.parametrize("capacity", [256, 2048])
@pytest.mark.parametrize("name", SHAPES)
def test_attentions_of_different_sizes(name, capacity, dtype):
    shape = SHAPES[name]
    w, ids = synthetic.random_hybrid_weights(shape, 3), torch.randint(0, 96, (212,), generator=torch.Generator().manual_seed(4))
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=capacity)
    mk, request = mk_kernel.get_mk(), RequestTable(g).open(0)
    got = torch.cat([decode_hybrid.run_tokens(g, mk, request, ids[i : i + 1], [0]) for i in range(len(ids))]).double().cpu()
    mk.check()
    want = (givopel_oracle if shape.plain else hybrid_oracle).forward(shape.to_config(), w, ids, dtype=torch.float64)
    d = got - want
    d = d - d.mean(-1, keepdim=True)
    err = float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max())
    assert err < TOLERANCE[shape.plain, dtype], f"{err:.3g}"
