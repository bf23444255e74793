"""The three bf16 parts of an fp32 value (csrc/qmk_hybrid_gemm.h, ``split2``) in the same arithmetic: exact from 2^-110 on, no further off than bf16's smallest
value below, each part of the value's sign and none above it."""
import numpy as np
import pytest


def parts_of(x):
    parts = []
    for _ in range(3):
        upper = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
        parts.append(upper)
        x = x - upper
    return parts


def values(exponent):
    bits = np.random.default_rng(exponent & 0xFFFF).integers(0, 1 << 23, 4096, dtype=np.uint32)
    bits[:4] = 0, 1, (1 << 23) - 1, 1 << 22
    x = (bits | np.uint32((exponent + 127) << 23)).view(np.float32)
    return np.concatenate((x, -x))


@pytest.mark.parametrize("exponent", [127, 100, 1, 0, -1, -60, -100, -109, -110])
def test_exact_over_the_range(exponent):
    x = values(exponent)
    parts = parts_of(x)
    assert np.array_equal(sum(p.astype(np.float64) for p in parts), x.astype(np.float64))
    assert all((np.sign(p) * np.sign(x) >= 0).all() and (np.abs(p) <= np.abs(x)).all() for p in parts)


@pytest.mark.parametrize("exponent", [-111, -120, -126, -127])
def test_cut_off_below(exponent):
    x = values(exponent)      # the last: values smaller than the smallest normal one
    short = np.abs(x.astype(np.float64) - sum(p.astype(np.float64) for p in parts_of(x)))
    assert 0 < short.max() < 2.0**-133
