"""The exact-weight GEMM over Q6_K rows, which the batched prefill runs
(gemm_q_f16_run of mxh_internal.h; no C entry takes Q6_K), at the edges of its
tiles, K splits and slabs (GPU).

Tiled rows (k a multiple of 2048) are read in place; rows in GGUF order are
regrouped first, their block count rounded up to eight, 64 MiB at a time in
equal pieces.  Outputs go into wider rows with a residual, as the model's do.
Reference and bound as in test_gemm_codes_gpu.py: the float64 product of the
decoded weights, within 2^-19 of sum_k |a_k w_k|.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import mxhip
import mxo

pytestmark = pytest.mark.gpu

vp, ci, cf = C.c_void_p, C.c_int, C.c_float


def symbol(name, args):
    f = getattr(mxhip.lib, name)
    f.restype, f.argtypes = ci, args
    return f


def gemm(type_, a, dw, n, k, form=mxo.FORM_REF, res=None, ldo=None):
    """[m, n] of the GEMM over rows at address dw, each output row ldo floats wide, with the guard columns."""
    rows = symbol("_ZN3mxh18rows_to_f16_launchEPKfiS1_fiPtS2_iS2_S2_iPfiP12ihipStream_t",
                  [vp, ci, vp, cf, ci, vp, vp, ci, vp, vp, ci, vp, ci, vp])
    run = symbol("_ZN3mxh14gemm_q_f16_runEiPKtS1_iS1_S1_iPKfPKvPfiS3_iiiiNS_9WorkspaceEP12ihipStream_t",
                 [ci, vp, vp, ci, vp, vp, ci, vp, vp, vp, ci, vp, ci, ci, ci, ci, ci, vp])
    m, ldo, st = len(a), ldo or n, vp(mxhip.lib.mxh_stream())
    da = mxhip.DeviceBuffer.from_array(a)
    hi, lo, sh, sl, sc = (mxhip.DeviceBuffer(b) for b in (2 * m * k, 2 * m * k, m * k // 16, m * k // 16, 4 * m))
    out = mxhip.DeviceBuffer.from_array(np.full((m, ldo), 7.0, np.float32))
    dr = mxhip.DeviceBuffer.from_array(np.pad(res, ((0, 0), (0, ldo - n)))) if res is not None else None
    assert rows(da.ptr, k, None, 0.0, k, hi.ptr, lo.ptr, k, sh.ptr, sl.ptr, k // 32, sc.ptr, m, st) == 0
    assert run(type_, hi.ptr, lo.ptr, k, sh.ptr, sl.ptr, k // 32, sc.ptr, dw, out.ptr, ldo, dr.ptr if dr else None, m, n,
               k, form, 0, st) == 0
    mxhip.synchronize()
    got = out.download(np.float32, m * ldo).reshape(m, ldo)
    for b in (da, hi, lo, sh, sl, sc, out, dr):
        if b is not None:
            b.close()
    return got


# (m, n, k): one row, each side of a tile of rows and of weight rows, one
# block, block counts not of eight, K splits of one and of odd numbers of blocks
SHAPES = [(1, 1, 256), (31, 255, 768), (8, 200, 4352), (33, 257, 2304), (65, 129, 6144), (129, 513, 2048),
          (200, 300, 5888), (257, 1030, 4096)]


@pytest.mark.parametrize("tiled", [False, True], ids=["gguf", "tiled"])
@pytest.mark.parametrize("m,n,k", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_q6k_edges(mxh, m, n, k, tiled):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    w = mxo.quantize(mxo.Q6_K, rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    a = rng.standard_normal((m, k), dtype=np.float32)
    a[0, :] *= 1e-4
    res = rng.standard_normal((m, n), dtype=np.float32) if m % 2 else None
    dw = mxhip.DeviceBuffer.from_array(w)
    t = mxhip.tile_rows(mxo.Q6_K, dw, n, k) if tiled else mxo.Q6_K
    if tiled and t == mxo.Q6_K:
        pytest.skip("no tiled layout for these rows")
    got = gemm(t, a, dw.ptr, n, k, res=res, ldo=n + 5)
    wd = mxo.dequant(mxo.Q6_K, w, n, k).astype(np.float64)
    want = a.astype(np.float64) @ wd.T
    # the residual is added in fp32: half a unit of the sum's last place
    bound = 2.0 ** -19 * (np.abs(a).astype(np.float64) @ np.abs(wd).T) + 1e-30
    if res is not None:
        want += res
        bound += 2.0 ** -24 * np.abs(want)
    err = np.abs(got[:, :n] - want)
    assert np.all(err <= bound), f"worst {float((err / bound).max()):.3g} x bound"
    assert np.all(got[:, n:] == 7.0)
    dw.close()


@pytest.mark.parametrize("m", [2, 130])
def test_q6k_more_than_one_slab(mxh, m):
    """10,000 rows of 57 blocks (13,440 bytes regrouped): 4,864 rows fit the
    slab, so three pieces of 3,584, 3,584 and 2,832.  A piece is planned for its
    own rows: its outputs are those of a call with these rows alone, bit for
    bit."""
    n, k, step = 10000, 14592, 3584
    rng = np.random.default_rng(m)
    raw = rng.integers(0, 256, (100, k // 256, 210), dtype=np.uint8)
    raw[:, :, 208:210] = (rng.standard_normal((100, k // 256, 1)) * 0.01).astype(np.float16).view(np.uint8)
    raw = raw.reshape(100, -1)
    # row i is pattern (7 i) % 100: the pieces' rows differ
    order = (7 * np.arange(n)) % 100
    dw = mxhip.DeviceBuffer.from_array(raw[order])
    a = rng.standard_normal((m, k), dtype=np.float32)
    res = rng.standard_normal((m, n), dtype=np.float32)
    got = gemm(mxo.Q6_K, a, dw.ptr, n, k, res=res, ldo=n + 3)
    wd = mxo.dequant(mxo.Q6_K, raw, 100, k).astype(np.float64)
    want = (a.astype(np.float64) @ wd.T)[:, order] + res
    bound = 2.0 ** -19 * (np.abs(a).astype(np.float64) @ np.abs(wd).T)[:, order] + 2.0 ** -24 * np.abs(want)
    assert np.all(np.abs(got[:, :n] - want) <= bound)
    assert np.all(got[:, n:] == 7.0)
    rb = k // 256 * 210
    for n0 in range(0, n, step):
        nn = min(step, n - n0)
        alone = gemm(mxo.Q6_K, a, dw.ptr + n0 * rb, nn, k, res=np.ascontiguousarray(res[:, n0:n0 + nn]), ldo=nn)
        assert np.array_equal(alone.view(np.uint32), np.ascontiguousarray(got[:, n0:n0 + nn]).view(np.uint32))
    dw.close()


def test_q6k_orders_give_the_same_bits_beyond_a_slab(mxh):
    """Rows that have a tiled order too (k a multiple of 2048): the pieces keep
    the K split of the call over all rows, which is that of the tiled rows."""
    m, n, k = 3, 10240, 14336
    rng = np.random.default_rng(9)
    raw = rng.integers(0, 256, (64, k // 256, 210), dtype=np.uint8)
    raw[:, :, 208:210] = (rng.standard_normal((64, k // 256, 1)) * 0.01).astype(np.float16).view(np.uint8)
    dw = mxhip.DeviceBuffer.from_array(np.tile(raw.reshape(64, -1), (n // 64, 1)))
    a = rng.standard_normal((m, k), dtype=np.float32)
    gguf = gemm(mxo.Q6_K, a, dw.ptr, n, k)
    t = mxhip.tile_rows(mxo.Q6_K, dw, n, k)
    assert t != mxo.Q6_K
    assert np.array_equal(gguf.view(np.uint32), gemm(t, a, dw.ptr, n, k).view(np.uint32))
    dw.close()
