"""Prefill attention where the keys are split among workgroups, and where the
running reference moves (GPU).

Few query tiles over many keys split the keys; parts of a tile may hold no key
of a row, or none of the tile (causal chunks from position 0).  Expected values
and the admitted error as in test_attention_prefill_gpu.py.
"""
from __future__ import annotations

import numpy as np
import pytest

import mxhip
from test_attention_prefill_gpu import reference

pytestmark = pytest.mark.gpu

# (nh, nkv, hd, p0, m): one query, a partial tile, odd groups, splits that end
# inside the chunk, tiles with fewer keys than the others
CASES = [(8, 1, 64, 2000, 1), (32, 8, 128, 1500, 16), (7, 1, 128, 640, 9), (3, 1, 32, 1023, 2), (8, 1, 128, 0, 300),
         (4, 4, 64, 0, 513), (14, 2, 64, 191, 65), (8, 8, 32, 64, 64)]


@pytest.mark.parametrize("kind", ["flat", "rising"])
@pytest.mark.parametrize("nh,nkv,hd,p0,m", CASES, ids=[f"h{a}-kv{b}-d{c}-p{d}-m{e}" for a, b, c, d, e in CASES])
def test_attention_splits(mxh, nh, nkv, hd, p0, m, kind):
    rng = np.random.default_rng(nh * 1000 + hd * 10 + p0 + m)
    n_ctx = p0 + m + 40
    q = rng.standard_normal((m, nh * hd)).astype(np.float32)
    kc = rng.standard_normal((n_ctx, nkv * hd)).astype(np.float16)
    if kind == "rising":  # scores grow with the key's position, by many powers of two over the row
        q = np.abs(q) * np.float32(0.5)
        kc = np.abs(kc) * np.linspace(0.0, 4.0, n_ctx, dtype=np.float16)[:, None]
    vc = rng.standard_normal((n_ctx, nkv * hd)).astype(np.float16)
    kc[p0 + m:] = np.float16(np.nan)
    vc[p0 + m:] = np.float16(np.nan)
    dq, dk, dv = (mxhip.DeviceBuffer.from_array(a) for a in (q, kc, vc))
    att = mxhip.DeviceBuffer.from_array(np.full(m * nh * hd, np.nan, np.float32))
    mxhip.attention_prefill(dq, dk, dv, att, p0, m, nh, nkv, hd)
    got = att.download(np.float32, m * nh * hd).reshape(m, nh * hd).astype(np.float64)
    want = reference(q, kc, vc, p0, m, nh, nkv, hd)
    bound = 1e-4 * float(np.abs(vc[: p0 + m].astype(np.float64)).max()) + 1e-4 * np.abs(want)
    err = np.abs(got - want)
    assert np.all(np.isfinite(got)), "non-finite output"
    assert np.all(err <= bound), f"worst {float((err / bound).max()):.3g} x bound"
    for b in (dq, dk, dv, att):
        b.close()


@pytest.mark.parametrize("nh,nkv,hd,p0,m", [(8, 2, 128, 200, 256), (8, 8, 64, 900, 256), (4, 1, 32, 3000, 64)],
                         ids=["whole", "d64", "split"])
def test_attention_probabilities_are_unbiased(mxh, nh, nkv, hd, p0, m):
    """With every V element 1 the outputs are sum(hi + lo of P) / sum(P): the
    split's own error.  Two halves rounded to nearest leave no mean error (a
    few 1e-9 over these rows, from the fp32 sums); a low half cut off instead
    lacks half a unit of its last place on average, with one sign: of P in
    [1, 2) that is 4/3 2^-23, -1.1e-7 at most.  2^-25 (3e-8) lies between.
    """
    rng = np.random.default_rng(hd + p0)
    q = rng.standard_normal((m, nh * hd)).astype(np.float32)
    kc = rng.standard_normal((p0 + m, nkv * hd)).astype(np.float16)
    vc = np.ones((p0 + m, nkv * hd), np.float16)
    dq, dk, dv = (mxhip.DeviceBuffer.from_array(a) for a in (q, kc, vc))
    att = mxhip.DeviceBuffer(4 * m * nh * hd)
    mxhip.attention_prefill(dq, dk, dv, att, p0, m, nh, nkv, hd)
    err = att.download(np.float32, m * nh * hd).astype(np.float64) - 1.0
    assert np.abs(err).max() <= 1e-6, f"worst {np.abs(err).max():.3g}"
    assert abs(err.mean()) <= 2.0 ** -25, f"mean error {err.mean():.3g}"
    for b in (dq, dk, dv, att):
        b.close()


def test_attention_near_equal_probabilities(mxh):
    """The rms error of single probabilities of nearly equal scores.  Scores are
    exact (one fp16 q value times one K value), V picks one key a dim.  exp2's
    last place, the split and the quotient leave 7.4e-8; an exponent rounded at
    a magnitude of 4 to 8 adds 2^-21 / sqrt(12) ln 2 = 9.5e-8: 1.2e-7 and more.
    """
    nh, nkv, hd, n = 8, 2, 128, 100
    qscale = np.float32(1.0) / np.sqrt(np.float32(hd)) * np.float32(1.4426950408889634)
    errs = []
    for seed in range(20):
        rng = np.random.default_rng(seed)
        c = np.float32(np.float16(1.0 + rng.random()))  # the scaled q the kernel is to see, exact in fp16
        near = np.float32(c / qscale)
        q0 = next(x for x in (near, np.nextafter(near, np.float32(9)), np.nextafter(near, np.float32(-9))) if x * qscale == c)
        q, kc, vc = np.zeros((1, nh, hd), np.float32), np.zeros((n, nkv, hd), np.float16), np.zeros((n, nkv, hd), np.float16)
        q[0, :, 5] = q0
        kc[:, :, 5] = 0.1 * rng.standard_normal((n, nkv))
        vc[np.arange(n), :, np.arange(n)] = 1
        dq, dk, dv = (mxhip.DeviceBuffer.from_array(a.reshape(len(a), -1)) for a in (q, kc, vc))
        att = mxhip.DeviceBuffer(4 * nh * hd)
        mxhip.attention_prefill(dq, dk, dv, att, n - 1, 1, nh, nkv, hd)
        got = att.download(np.float32, nh * hd).reshape(nh, hd)[:, :n].astype(np.float64)
        p = 2.0 ** (float(c) * kc[:, :, 5].astype(np.float64))
        errs.append(got / np.repeat((p / p.sum(0)).T, nh // nkv, axis=0) - 1)
        for b in (dq, dk, dv, att):
            b.close()
    rms = float(np.sqrt(np.mean(np.square(errs))))
    assert rms <= 1e-7, f"rms error {rms:.3g}"


@pytest.mark.parametrize("nh,nkv,hd,p0,m", [(8, 2, 128, 0, 300), (8, 8, 64, 500, 100), (4, 1, 32, 3000, 64)],
                         ids=["d128", "d64", "split"])
def test_attention_error_is_that_of_22_bits(mxh, nh, nkv, hd, p0, m):
    """2-norm error against float64 at ordinary scores.  q as fp16 hi + lo is
    off by 2^-23 of itself at most, a score (in base 2, |s| about 1.4) by about
    as much of its terms: 2e-7 to 5e-7 of the outputs with the sums.  One q in
    some thousand with halves that do not belong together (2^-12 off) made it
    4e-6 to 1.2e-5.  2^-20 (9.5e-7) lies between.
    """
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((m, nh * hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((p0 + m, nkv * hd)).astype(np.float16) for _ in range(2))
    dq, dk, dv = (mxhip.DeviceBuffer.from_array(a) for a in (q, kc, vc))
    att = mxhip.DeviceBuffer(4 * m * nh * hd)
    mxhip.attention_prefill(dq, dk, dv, att, p0, m, nh, nkv, hd)
    got = att.download(np.float32, m * nh * hd).reshape(m, nh * hd).astype(np.float64)
    want = reference(q, kc, vc, p0, m, nh, nkv, hd)
    rel = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert rel <= 2.0 ** -20, f"relative error {rel:.3g}"
    for b in (dq, dk, dv, att):
        b.close()
