"""mxh_matmul_rhs_t over several rows against one mxh_gemv per row (GPU).

A call takes its rows eight, four or two at a time (as many as the LDS holds)
and a last one alone; each meets the weights in the GEMV's own arithmetic and
order, so the results are required to be the GEMV's bit for bit (the GEMV
itself is held to the oracle in test_gemv_gpu.py).
"""
from __future__ import annotations

import numpy as np
import pytest

import mxhip
import mxo

pytestmark = pytest.mark.gpu

TYPES = {"F32": mxo.F32, "F16": mxo.F16, "Q8_0": mxo.Q8_0, "Q5_0": mxo.Q5_0, "Q4_K": mxo.Q4_K, "Q5_K": mxo.Q5_K,
         "Q6_K": mxo.Q6_K}
# (m, n, k): every count of rows per launch and its remainders; one weight row,
# a wave's, more than the chip's waves; one block, part of a step, the longest
SHAPES = [(2, 1, 256), (3, 33, 512), (4, 300, 2304), (5, 513, 4096), (7, 64, 768), (8, 4100, 256), (9, 17, 2048),
          (11, 40, 14336), (17, 129, 1024), (2, 6, 15360)]


@pytest.mark.parametrize("tiled", [False, True], ids=["gguf", "tiled"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("name", list(TYPES))
def test_matmul_rows_equal_gemvs(mxh, name, m, n, k, tiled):
    t = TYPES[name]
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    if name in ("Q8_0", "Q5_0", "F16", "F32") and k == 768:
        k = 736  # whole blocks of 32 only
    wf = rng.standard_normal((n, k), dtype=np.float32)
    w = wf if name == "F32" else wf.astype(np.float16) if name == "F16" else mxo.quantize(t, wf)
    x = rng.standard_normal((m, k), dtype=np.float32)
    x[0] *= 1e-4
    dw, dx = mxhip.DeviceBuffer.from_array(w), mxhip.DeviceBuffer.from_array(x)
    tt = mxhip.tile_rows(t, dw, n, k) if tiled else t
    if tiled and tt == t:
        pytest.skip("no tiled layout for these rows")
    # a guard behind the output: nothing may be written past m x n
    out = mxhip.DeviceBuffer.from_array(np.full(m * n + 64, 7.0, np.float32))
    ref = mxhip.DeviceBuffer.from_array(np.zeros(m * n, np.float32))
    form = mxo.FORM_GGML if m % 2 else mxo.FORM_REF
    assert mxhip.lib.mxh_matmul_rhs_t(tt, dx.ptr, m, dw.ptr, n, k, out.ptr, form) == 0
    for i in range(m):
        assert mxhip.lib.mxh_gemv(tt, dw.ptr, dx.ptr + 4 * i * k, ref.ptr + 4 * i * n, n, k, form) == 0
    mxhip.synchronize()
    got = out.download(np.float32, m * n + 64)
    assert np.array_equal(got[:m * n], ref.download(np.float32, m * n))
    assert np.all(got[m * n:] == 7.0)
    for b in (dw, dx, out, ref):
        b.close()


# long fp32 and fp16 rows: one weight row a wave up to eight per CU, two above
@pytest.mark.parametrize("m,n,k", [(2, 2048, 4128), (3, 2049, 4128), (5, 257, 4096), (9, 300, 5024), (5, 7, 14336)])
@pytest.mark.parametrize("name", ["F16", "F32"])
def test_long_float_rows_equal_gemvs(mxh, name, m, n, k):
    test_matmul_rows_equal_gemvs(mxh, name, m, n, k, False)
