"""The device sampler's selection at its edges (GPU): group sizes, ties,
candidates that do not fit the sort, NaN and infinities, against the oracle's
sampler (the same id for the same logits and draw).
"""
from __future__ import annotations

import numpy as np
import pytest

import mxhip
import mxo

pytestmark = pytest.mark.gpu


def logits_of(kind, n):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 2.0).astype(np.float32)
    if kind == "equal":  # every key ties: the lowest ids
        x[:] = 0.5
    elif kind == "sorted":  # the top k side by side, at the end (a tail group)
        x = np.sort(x)
    elif kind == "block":  # 20,000 large logits side by side, few distinct
        x[n // 3:n // 3 + min(n // 2, 20000)] = 9.0 + np.float32(0.125) * rng.integers(0, 3, min(n // 2, 20000))
    elif kind == "inf":
        x[rng.random(n) < 0.7] = -np.inf
    elif kind == "neg":
        x = -np.abs(x) - 1
    return x


# one id, one group's edges, each group size's range, the tail of a group
SIZES = [1, 5, 4097, 49153, 98304, 151936, 200003]


@pytest.mark.parametrize("k", [1, 40, 1000, 4096])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["normal", "equal", "sorted", "block", "inf", "neg"])
def test_sample_selection(mxh, kind, n, k):
    k = min(k, n)
    x = logits_of(kind, n)
    buf = mxhip.DeviceBuffer.from_array(x)
    for t, p, mp in ((1.3, 1.0, 0.0), (0.9, 0.97, 0.01)):
        state = seed = 0xD0E5 + k
        for d in range(4):
            want, state = mxo.sample(x, k, t, p, mp, state)
            got = mxhip.sample(buf, n, k, t, p, mp, seed, d)
            assert got == want, f"T {t} draw {d}: device {got}, oracle {want}"
    buf.close()


def test_sample_nan_last(mxh):
    """NaN logits rank below every number: with enough numbers they are never drawn."""
    n = 30001
    x = np.full(n, np.nan, np.float32)
    good = np.random.default_rng(3).choice(n, 50, replace=False)
    x[good] = np.linspace(-3, 3, 50, dtype=np.float32)
    buf = mxhip.DeviceBuffer.from_array(x)
    clean = np.where(np.isnan(x), np.float32(-np.inf), x)
    state = 11
    for d in range(8):
        want, state = mxo.sample(clean, 50, 1.5, 1.0, 0.0, state)
        assert mxhip.sample(buf, n, 50, 1.5, 1.0, 0.0, 11, d) == want
    buf.close()
