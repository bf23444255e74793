"""The residual's streams behind a prefill product (csrc/qmk_hybrid_gemm.h, ResidualQuads): up to four streams several quads at a time, more of them one by one, on
tiles that tokens and rows of weights do not divide; against the plain implementation in 64 bits, tolerances as in test_gpu_hybrid_products.py."""
import pytest
import torch

import hybrid_oracle
from qimeng_megakernel_amd import decode_hybrid, synthetic
from qimeng_megakernel_amd.decode_schedule_hybrid import mk_kernel, weights
from qimeng_megakernel_amd.decode_schedule_hybrid.globs import build_globals
from qimeng_megakernel_amd.decode_schedule_hybrid.state import RequestTable

pytestmark = pytest.mark.gpu

DEVICE = "cuda:0"
TOL = {torch.float32: 2e-5, torch.bfloat16: 4e-2}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("n", [20, 150, 700])
@pytest.mark.parametrize("streams", [1, 3, 4, 5, 8])
def test_streams_of_any_number(streams, n, dtype):
    shape = synthetic.hybrid_shape("a", width=1104, vocab=96, streams=streams, ff={"a": 1536}, heads=2, dim=64, rot_dim=32, v_dim=64, rank=64, window=100)
    w = synthetic.random_hybrid_weights(shape, 3, DEVICE)
    tokens = torch.randint(0, shape.vocab, (n,), generator=torch.Generator().manual_seed(5))
    with torch.device(DEVICE):
        want = hybrid_oracle.forward(shape.to_config(), w, tokens.to(DEVICE), dtype=torch.float64)
    g = build_globals(shape, weights.pack(shape, w, DEVICE), dtype=dtype, max_positions=n, portion_rows=n)
    got = decode_hybrid.run_tokens(g, mk_kernel.get_mk(), RequestTable(g).open(0), tokens, range(n)).double()
    d = got - want
    d = d - d.mean(-1, keepdim=True)
    err = float((d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()).max())
    assert err < TOL[dtype], f"{err:.3g}"
