"""mxh_dequant at the edges of its work split and at odd addresses (GPU).

A thread decodes four elements and a workgroup 4,096; the rows may start at any
byte address and the output at any float.  Results are the oracle's bit for
bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import mxhip
import mxo

pytestmark = pytest.mark.gpu

TYPES = {"F32": mxo.F32, "F16": mxo.F16, "Q8_0": mxo.Q8_0, "Q5_0": mxo.Q5_0, "Q4_K": mxo.Q4_K, "Q5_K": mxo.Q5_K,
         "Q6_K": mxo.Q6_K}
# one block, one short of and one past a workgroup's elements, several workgroups
SHAPES = [(1, 256), (3, 1280), (1, 4096), (17, 256), (9, 4352)]


@pytest.mark.parametrize("offset", [0, 1, 2, 4], ids=lambda o: f"at{o}")
@pytest.mark.parametrize("rows,cols", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("name", list(TYPES))
def test_dequant_edges(mxh, name, rows, cols, offset):
    t = TYPES[name]
    if name not in ("Q4_K", "Q5_K", "Q6_K") and rows == 3:
        cols = 1248  # whole blocks of 32 only
    rng = np.random.default_rng(rows + cols + offset)
    wf = rng.standard_normal((rows, cols), dtype=np.float32)
    raw = wf if name == "F32" else wf.astype(np.float16) if name == "F16" else mxo.quantize(t, wf)
    raw = np.ascontiguousarray(raw).view(np.uint8).reshape(-1)
    dw = mxhip.DeviceBuffer.from_array(np.concatenate([np.zeros(offset, np.uint8), raw]))
    n = rows * cols
    out = mxhip.DeviceBuffer.from_array(np.full(n + 64, 7.0, np.float32))
    first = 1 if offset else 0  # the output's first float
    form = mxo.FORM_GGML if rows % 2 else mxo.FORM_REF
    assert mxhip.lib.mxh_dequant(t, dw.ptr + offset, out.ptr + 4 * first, rows, cols, form) == 0
    mxhip.synchronize()
    got = out.download(np.float32, n + 64)
    want = mxo.dequant(t, raw, rows, cols, form).reshape(-1)
    assert np.array_equal(got[first:first + n].view(np.uint32), want.view(np.uint32))
    assert np.all(got[:first] == 7.0) and np.all(got[first + n:] == 7.0)
    dw.close()
    out.close()
