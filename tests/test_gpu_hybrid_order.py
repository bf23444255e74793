"""bf16 portions are computed in one order whatever their length: a token's logits are the same bits in a portion of any length that starts at the
same place.  (Lengths at which the tiles of the products change; no recurrence whose scan is cut by the length.)"""
import pytest
import torch

from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu

MOST = 2100
LENGTHS = (2, 33, 64, 65, 129, 200, 257, 520, 1023, 1025, 1531, 2049)
SHAPES = {
    "streams": synthetic.hybrid_shape("aw", width=2048, vocab=512, streams=2, ff={"a": 4096, "w": 2816}, heads=8, dim=128, rot_dim=64, v_dim=128, rank=256, window=300,
                                      wkv_heads=16, wkv_dim=64, wkv_rank=64),
    "ragged": synthetic.hybrid_shape("aw", width=1104, vocab=336, streams=3, ff={"a": 1744}, heads=3, dim=80, rot_dim=32, v_dim=112, rank=144, window=77,
                                     wkv_heads=5, wkv_dim=40, wkv_rank=12),
    "plain": synthetic.looped_shape("pgp", width=2048, vocab=512, ff={"p": 4096}, loop=(1, 2, 2), heads=4, kv_heads=2, delta_heads=4, delta_kv_heads=2, gla_heads=2),
    "large heads": synthetic.looped_shape("pg", width=256, vocab=96, heads=2, kv_heads=1, dim=200, v_dim=250, rot_dim=36, delta_heads=2, delta_kv_heads=2, delta_dim=250,
                                          delta_v_dim=136, delta_rank=24, gate_rank=8, gla_heads=2, gla_dim=136, gla_v_dim=250, gla_rank=24),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_a_tokens_bits_do_not_depend_on_its_portions_length(name):
    shape = SHAPES[name]
    g = build_globals(shape, weights.pack(shape, synthetic.random_hybrid_weights(shape, 3, "cuda"), "cuda:0"), dtype=torch.bfloat16, max_positions=MOST + 8, portion_rows=MOST)
    mk, table = mk_kernel.get_mk(), RequestTable(g)
    tokens = torch.randint(0, shape.vocab, (MOST,), generator=torch.Generator().manual_seed(5))

    def logits(n):
        request = table.open(n)
        got = decode_hybrid.run_tokens(g, mk, request, tokens[:n], range(n))
        table.close(n)
        return got

    whole = logits(MOST)
    for n in LENGTHS:
        differing = int((logits(n) != whole[:n]).any(-1).sum())
        assert differing == 0, f"{differing} of {n} tokens"
