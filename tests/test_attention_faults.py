"""What the GPU test of the prefill's bf16 attention can see: mistakes at a window's or a stage's edge, planted in the plain implementation, move the logits of its
inputs by more than twice its tolerance on every shape."""
import math

import pytest
import torch

import givopel_oracle
import hybrid_oracle
from test_gpu_hybrid_attention import MOST, SHAPES, inputs, tolerance, worst

DIST = torch.arange(MOST)[:, None] - torch.arange(MOST)[None, :]
KEY = torch.arange(MOST)[None, :].expand(MOST, MOST)
#: which keys a query sees, by mistake
FAULTS = {
    "a key too many at the window's end": lambda window: (DIST >= 0) & (DIST <= window),
    "a key too few at the window's end": lambda window: (DIST >= 0) & (DIST < window - 1),
    "the next key": lambda window: (DIST >= -1) & (DIST < window),
    "without the last of every 32 keys": lambda window: (DIST >= 0) & (DIST < window) & ((KEY % 32 != 31) | (DIST == 0)),
    "without the first of every 64 keys": lambda window: (DIST >= 0) & (DIST < window) & ((KEY % 64 != 0) | (DIST == 0)),
}


def attention(seen_by):
    def attend(q, k, v, scale, window=MOST):
        out, seen, group = [], seen_by(window), q.shape[1] // k.shape[1]
        for head in range(q.shape[1]):
            s = torch.where(seen, (q[:, head] @ k[:, head // group].T) * scale, -math.inf)
            out.append(torch.softmax(s, -1) @ v[:, head // group])
        return torch.stack(out, dim=1)

    return attend


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_a_mistake_at_an_edge_is_outside_the_tolerance(monkeypatch, name):
    shape, w, tokens = inputs(name)
    oracle, mechanism = (givopel_oracle, "causal_attention") if shape.plain else (hybrid_oracle, "windowed_softmax_attention")

    def forward(seen_by=None):
        with monkeypatch.context() as planted:
            if seen_by is not None:
                planted.setattr(oracle, mechanism, attention(seen_by))
            return oracle.forward(shape.to_config(), w, tokens, dtype=torch.float64)

    want = forward()
    assert worst(forward(lambda window: (DIST >= 0) & (DIST < window)), want) < 1e-9
    for fault, seen_by in FAULTS.items():
        if "window" not in fault or not shape.plain:
            assert worst(forward(seen_by), want) > 2 * tolerance(shape), fault
