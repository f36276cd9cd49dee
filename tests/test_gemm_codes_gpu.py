"""The pipelined exact-weight GEMM (mxh_gemm_q_f16) at the edges of its tiles,
K blocks and split K (GPU).

Tiles are 32, 64 or 128 activation rows by 128 or 256 weight rows, K advances
in 256-element blocks that the K splits share out unevenly, tiled rows end in
partial tiles of 16 (Q4_K), 8 (Q5_K) or 64 (Q8_0) blocks, and Q8_0 / Q5_0 rows
in GGUF order are regrouped first.  Reference and bound as in
test_prefill_gpu.py: the float64 product of the exactly decoded weights,
within 2^-19 of sum_k |a_k w_k| (22-bit activations, fp32 sums).
"""
from __future__ import annotations

import numpy as np
import pytest

import mxhip
import mxo

pytestmark = pytest.mark.gpu

TYPES = {"Q4_K": mxo.Q4_K, "Q5_K": mxo.Q5_K, "Q8_0": mxo.Q8_0, "Q5_0": mxo.Q5_0}
# (m, n, k): one row, each side of a tile of rows, of weight rows and of K
SHAPES = [(1, 1, 256), (31, 255, 512), (33, 257, 768), (64, 129, 4352), (65, 513, 2304), (129, 256, 4096),
          (200, 300, 2816), (257, 1030, 5120)]


@pytest.mark.parametrize("tiled", [False, True], ids=["gguf", "tiled"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("name", list(TYPES))
def test_gemm_codes_edges(mxh, name, m, n, k, tiled):
    t = TYPES[name]
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    w = mxo.quantize(t, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    a = rng.standard_normal((m, k), dtype=np.float32)
    a[0, :] *= 1e-4
    form = mxo.FORM_GGML if k % 512 else mxo.FORM_REF
    dw, da = mxhip.DeviceBuffer.from_array(w), mxhip.DeviceBuffer.from_array(a)
    # a guard behind the output: nothing may be written past m x n
    out = mxhip.DeviceBuffer.from_array(np.full(m * n + 64, 7.0, np.float32))
    tt = mxhip.tile_rows(t, dw, n, k) if tiled else t
    mxhip.gemm_f16(tt, da, m, dw, n, k, out, form)
    got = out.download(np.float32, m * n + 64)
    wd = mxo.dequant(t, w, n, k, form).astype(np.float64)
    bound = 2.0 ** -19 * (np.abs(a).astype(np.float64) @ np.abs(wd).T) + 1e-30
    err = np.abs(got[:m * n].reshape(m, n) - a.astype(np.float64) @ wd.T)
    assert np.all(err <= bound), f"worst {float((err / bound).max()):.3g} x bound"
    assert np.all(got[m * n:] == 7.0)
    for b in (dw, da, out):
        b.close()
