"""The work a program has this library do, as measurable cases.

Every case is one pass through the public entry points on data in HBM, as a
local-LLM runtime calls them:

- ``model``      a whole call on a GGUF model: reset, prefill a prompt, then
                 single-token steps whose logits come back to the host (a
                 runtime with its own sampler, teacher-forced here so that a
                 pass does not depend on near-ties);
- ``gemv``       one token's walk over a layer stack's projections of one
                 shape: `count` distinct weight matrices, one GEMV each;
- ``rows``       ``mxh_matmul_rhs_t``: the same projection for a few rows at
                 once (a short prompt, a small batch);
- ``gemm``       ``mxh_gemm_q_f16``: a prompt chunk's projection on the
                 matrix cores;
- ``attention``  ``mxh_attention_prefill``: causal attention of a prompt chunk
                 over the fp16 K/V cache;
- ``dequant``    ``mxh_dequant``: GGUF rows to fp32;
- ``sample``     ``mxh_sample``: one sampling decision over device logits.

Weights are quantized normal weights in the GGUF block formats (the layouts
of the published formats, packed below), activations are normal with a few
large channels, as the outputs of a norm are.
"""
import ctypes
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("minxfmr.cpp_amd"))
import mxhip  # noqa: E402

TYPES = {"F32": mxhip.F32, "F16": mxhip.F16, "Q5_0": mxhip.Q5_0, "Q8_0": mxhip.Q8_0, "Q4_K": mxhip.Q4_K,
         "Q5_K": mxhip.Q5_K, "Q6_K": mxhip.Q6_K}
# the architectures of the benchmark and the full-size tests (layer counts per case)
ARCHS = {
    "qwen3-0.6b": dict(arch="qwen3", n_embd=1024, n_head=16, n_head_kv=8, head_dim=128, n_ff=3072, n_vocab=151936,
                       rope_theta=1e6, eps=1e-6, qk_norm=True, tied=True),
    "qwen3-8b": dict(arch="qwen3", n_embd=4096, n_head=32, n_head_kv=8, head_dim=128, n_ff=12288, n_vocab=151936,
                     rope_theta=1e6, eps=1e-6, qk_norm=True, tied=False),
    "llama3-8b": dict(arch="llama", n_embd=4096, n_head=32, n_head_kv=8, head_dim=128, n_ff=14336, n_vocab=128256,
                      rope_theta=5e5, eps=1e-5, qk_norm=False, tied=False),
}
# weight types of a file: projections, attn_v and ffn_down, lm-head, embedding
MIXES = {"q8_0": ("Q8_0", "Q8_0", "Q8_0", "Q8_0"), "q4_k": ("Q4_K", "Q4_K", "Q8_0", "Q4_K"),
         "q4_k+q5_k": ("Q4_K", "Q5_K", "Q8_0", "Q4_K"), "q4_k_m": ("Q4_K", "Q6_K", "Q6_K", "Q4_K")}


def listed():
    return [
        # a small chat model at a short prompt: 28 thin layers, where launches and latency count
        dict(name="model-qwen3-0.6b-q8", op="model", arch="qwen3-0.6b", mix="q8_0", layers=28, n_ctx=160, prompt=32,
             steps=8),
        # a Q4_K_M-style file (the usual download) at 8B widths, a prompt of more than one chunk, a 4K context
        dict(name="model-llama3-8b-q4km", op="model", arch="llama3-8b", mix="q4_k_m", layers=3, n_ctx=4096,
             prompt=700, steps=4),
        # decode: the smallest call, one o-projection of the 0.6B model
        dict(name="gemv-1024x2048-q8", op="gemv", type="Q8_0", tiled=True, n=1024, k=2048, count=1, form=0),
        # decode: the widest projection of an 8B layer, over eight layers (weights beyond every cache)
        dict(name="gemv-24576x4096-q4k", op="gemv", type="Q4_K", tiled=True, n=24576, k=4096, count=8, form=0),
        # decode: the 8B lm-head
        dict(name="gemv-151936x4096-q8", op="gemv", type="Q8_0", tiled=True, n=151936, k=4096, count=1, form=0),
        # a few rows at once (a small batch) through one 8B projection, weights as the file holds them
        dict(name="rows-8x4096x4096-q4k", op="rows", type="Q4_K", tiled=False, m=8, n=4096, k=4096, form=0),
        # prefill: a full chunk through the widest projection of an 8B layer
        dict(name="gemm-512x24576x4096-q4k", op="gemm", type="Q4_K", tiled=True, m=512, n=24576, k=4096, form=0),
        # prefill: one row past a tile, the long rows of a mixed file's down projection
        dict(name="gemm-129x4096x14336-q5k", op="gemm", type="Q5_K", tiled=True, m=129, n=4096, k=14336, form=0),
        # prefill: a short prompt through the 0.6B gate|up
        dict(name="gemm-31x6144x1024-q8", op="gemm", type="Q8_0", tiled=True, m=31, n=6144, k=1024, form=0),
        # prefill: a chunk late in a long prompt
        dict(name="attention-512-at-7680", op="attention", m=512, p0=7680, nh=32, nkv=8, hd=128),
        # weights widened to fp32, as a runtime does for an op it runs itself
        dict(name="dequant-4096x14336-q6k", op="dequant", type="Q6_K", rows=4096, cols=14336, form=0),
        # one sampled token over a full vocabulary
        dict(name="sample-151936-k40", op="sample", n=151936, top_k=40, temperature=0.7, top_p=0.95, min_p=0.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, lo, hi, unit=256):
    return min(hi, max(lo, _log(rng, lo, hi) // unit * unit))


def draw(rng):
    op = rng.choice(["model", "gemv", "gemv", "rows", "rows", "gemm", "gemm", "gemm", "attention", "attention",
                     "dequant", "sample"])
    form = rng.choice([0, 0, 1])
    if op == "model":
        arch = rng.choice(list(ARCHS))
        mix = "q8_0" if arch == "qwen3-0.6b" else rng.choice(["q4_k", "q4_k+q5_k", "q4_k_m"])
        prompt = _log(rng, 4, 700)
        return dict(op=op, arch=arch, mix=mix, layers=rng.randint(1, 3), n_ctx=rng.choice([prompt + 16, 1024, 4096]),
                    prompt=prompt, steps=rng.randint(1, 4))
    if op == "gemv":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q8_0", "Q5_0", "F16", "F32"])
        n, k = _log(rng, 256, 40000), _cols(rng, 512, 14336)
        count = max(1, min(8, int(3e8 / (n * k))))
        return dict(op=op, type=t, tiled=t in ("Q4_K", "Q5_K", "Q6_K", "Q8_0") and rng.random() < 0.75, n=n, k=k,
                    count=count, form=form)
    if op == "rows":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q8_0", "Q5_0", "F16", "F32"])
        m, k = _log(rng, 2, 96), _cols(rng, 512, 14336)
        n = min(_log(rng, 256, 25000), max(256, int(4e9 / (m * k))))
        return dict(op=op, type=t, tiled=t in ("Q4_K", "Q5_K", "Q6_K", "Q8_0") and rng.random() < 0.5, m=m, n=n, k=k,
                    form=form)
    if op == "gemm":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q8_0", "Q8_0", "Q5_0"])
        m, k = _log(rng, 2, 600), _cols(rng, 512, 14336)
        n = min(_log(rng, 512, 30000), int(5e10 / (m * k)))
        return dict(op=op, type=t, tiled=t != "Q5_0" and rng.random() < 0.75, m=m, n=n, k=k, form=form)
    if op == "attention":
        nkv, group, hd = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 3, 4, 7, 8]), rng.choice([32, 64, 128, 128])
        m, p0 = _log(rng, 2, 512), rng.choice([0, 0, _log(rng, 16, 7680)])
        return dict(op=op, m=m, p0=p0, nh=nkv * group, nkv=nkv, hd=hd)
    if op == "dequant":
        t = rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q5_0", "F16"])
        cols = _cols(rng, 256, 14336)
        return dict(op=op, type=t, rows=min(_log(rng, 16, 30000), int(1e8 / cols)), cols=cols, form=form)
    n = _log(rng, 30000, 160000)
    return dict(op=op, n=n, top_k=_log(rng, 1, 1000), temperature=round(rng.uniform(0.5, 1.5), 3),
                top_p=round(rng.uniform(0.8, 1.0), 3), min_p=rng.choice([0.0, 0.02, 0.1]))


# ---- weights in the GGUF block formats -------------------------------------------------


def _bytes(t, shape):
    return t.contiguous().view(torch.uint8).reshape(*shape, -1)


def _safe(d):
    return torch.where(d == 0, torch.ones_like(d), d)


def quantize(w, name):
    """[rows, cols] fp32 weights as the rows' raw blocks, [rows, bytes] uint8."""
    rows, cols = w.shape
    if name in ("F32", "F16"):
        return _bytes(w if name == "F32" else w.half(), (rows,))
    if name == "Q8_0":
        x = w.reshape(rows, -1, 32)
        d = (x.abs().amax(-1, keepdim=True) / 127).half()
        q = (x / _safe(d.float())).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d, x.shape[:2]), _bytes(q, x.shape[:2])], -1).reshape(rows, -1)
    if name == "Q5_0":
        x = w.reshape(rows, -1, 32)
        top = x.gather(-1, x.abs().argmax(-1, keepdim=True))
        d = (top / -16).half()
        q = ((x / _safe(d.float())).round() + 16).clamp(0, 31).to(torch.int64)
        qh = ((q >> 4) << torch.arange(32, device=w.device)).sum(-1, keepdim=True).to(torch.int32)
        qs = ((q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)).to(torch.uint8)
        return torch.cat([_bytes(d, x.shape[:2]), _bytes(qh, x.shape[:2]), qs], -1).reshape(rows, -1)
    nb = (rows, cols // 256)
    if name in ("Q4_K", "Q5_K"):
        levels = 15 if name == "Q4_K" else 31
        x = w.reshape(*nb, 8, 32)
        m = -x.amin(-1).clamp(max=0)
        sc = (x.amax(-1) + m) / levels
        d, dm = (sc.amax(-1, keepdim=True) / 63).half(), (m.amax(-1, keepdim=True) / 63).half()
        ls = (sc / _safe(d.float())).round().clamp(0, 63).to(torch.uint8)
        lm = (m / _safe(dm.float())).round().clamp(0, 63).to(torch.uint8)
        ds = _safe(d.float() * ls)
        q = ((x + (dm.float() * lm).unsqueeze(-1)) / ds.unsqueeze(-1)).round().clamp(0, levels).to(torch.uint8)
        scales = torch.cat([ls[..., :4] | (ls[..., 4:] >> 4 << 6), lm[..., :4] | (lm[..., 4:] >> 4 << 6),
                            (ls[..., 4:] & 15) | ((lm[..., 4:] & 15) << 4)], -1)
        q2 = q.reshape(*nb, 4, 2, 32)
        qs = ((q2[..., 0, :] & 15) | ((q2[..., 1, :] & 15) << 4)).reshape(*nb, 128)
        parts = [_bytes(d, nb), _bytes(dm, nb), scales]
        if name == "Q5_K":
            parts.append(sum((q[..., j, :] >> 4) << j for j in range(8)))
        return torch.cat(parts + [qs], -1).reshape(rows, -1)
    assert name == "Q6_K"
    x = w.reshape(*nb, 16, 16)
    s = x.gather(-1, x.abs().argmax(-1, keepdim=True)).squeeze(-1) / -32
    d = (s.abs().amax(-1, keepdim=True) / 127).half()
    sc = (s / _safe(d.float())).round().clamp(-128, 127).to(torch.int8)
    ds = _safe(d.float() * sc)
    q = ((x / ds.unsqueeze(-1)).round().clamp(-32, 31) + 32).to(torch.uint8).reshape(*nb, 2, 4, 32)
    ql = torch.cat([(q[..., 0:2, :] & 15) | ((q[..., 2:4, :] & 15) << 4)], -1).reshape(*nb, 128)
    qh = sum((q[..., g, :] >> 4) << (2 * g) for g in range(4)).reshape(*nb, 64)
    return torch.cat([ql, qh, _bytes(sc, nb), _bytes(d, nb)], -1).reshape(rows, -1)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def decode(raw, name, form=0):
    """Raw block rows [rows, bytes] as float64 weights [rows, cols]; form 0 / 1: the two 6-bit scale unpackings."""
    rows = raw.shape[0]
    if name in ("F32", "F16"):
        return raw.contiguous().view(torch.float32 if name == "F32" else torch.float16).double()
    size = {"Q8_0": 34, "Q5_0": 22, "Q4_K": 144, "Q5_K": 176, "Q6_K": 210}[name]
    b = raw.reshape(rows, -1, size)
    if name == "Q8_0":
        return (_half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8)).reshape(rows, -1)
    if name == "Q5_0":
        qh = b[..., 2:6].contiguous().view(torch.int32).long()
        hi = (qh >> torch.arange(32, device=raw.device)) & 1
        q = torch.cat([b[..., 6:] & 15, b[..., 6:] >> 4], -1).long() | (hi << 4)
        return (_half(b[..., :2]) * (q - 16)).reshape(rows, -1)
    if name in ("Q4_K", "Q5_K"):
        s = b[..., 4:16]
        top = s[..., 0:4] if form else s[..., 4:8]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (top >> 6 << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
        qs = b[..., -128:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], -2).reshape(rows, -1, 8, 32)
        if name == "Q5_K":
            q = q | (torch.stack([(b[..., 16:48] >> j) & 1 for j in range(8)], -2) << 4)
        d, dm = _half(b[..., :2]), _half(b[..., 2:4])
        return ((d * sc).unsqueeze(-1) * q - (dm * mn).unsqueeze(-1)).reshape(rows, -1)
    ql, qh = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 32)
    q = torch.cat([ql & 15, ql >> 4], -2) | (torch.stack([(qh >> (2 * g)) & 3 for g in range(4)], -2) << 4)
    sc = b[..., 192:208].contiguous().view(torch.int8).double() * _half(b[..., 208:210])
    return (sc.unsqueeze(-1) * (q.double() - 32).reshape(rows, -1, 16, 16)).reshape(rows, -1)


# ---- inputs ----------------------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator("cuda").manual_seed((seed * 1000003 + salt) & 0x7FFFFFFF)


def _normal(shape, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _activations(shape, g):
    """Normal values, one channel in 64 eight times as large."""
    big = torch.rand(shape[-1], generator=g, device="cuda") < 1 / 64
    return _normal(shape, g) * (1 + 7 * big)


def _raw(name, rows, cols, seed, salt, slack=256):
    """A quantized N(0, 0.02) matrix in its own allocation, as uint8 [rows, bytes] (`slack` bytes behind it)."""
    g = _gen(seed, salt)
    width = mxhip.row_bytes(TYPES[name], cols)
    buf = torch.empty(rows * width + slack, dtype=torch.uint8, device="cuda")
    out = buf[: rows * width].view(rows, width)
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        out[r:r + step] = quantize(0.02 * _normal((min(step, rows - r), cols), g), name)
    return out


def _matvec_inputs(case, seed):
    name, n, k = case["type"], case["n"], case["k"]
    ws = [_raw(name, n, k, seed, 10 + i) for i in range(case.get("count", 1))]
    x = _activations((case.get("m", 1), k), _gen(seed, 1))
    return ws, x


def _model_file(case, seed):
    a = dict(ARCHS[case["arch"]])
    w, vd, out, embd = (TYPES[t] for t in MIXES[case["mix"]])
    f = tempfile.NamedTemporaryFile(suffix=".gguf", delete=False)
    f.close()
    mxhip.write_synthetic_gguf(f.name, a.pop("arch"), n_layer=case["layers"], ctx=40960, wtype=w, attn_v_type=vd,
                               ffn_down_type=vd, out_type=out, embd_type=embd, seed=seed,
                               threads=min(16, os.cpu_count() or 8), **a)
    return f.name


def _model_ids(case, seed):
    rng = np.random.default_rng(seed + 1)
    n = ARCHS[case["arch"]]["n_vocab"]
    return rng.integers(0, n, case["prompt"]).astype(np.int32), rng.integers(0, n, case["steps"]).astype(np.int32)


def _attention_inputs(case, seed):
    rows, kvd = case["p0"] + case["m"], case["nkv"] * case["hd"]
    q = 2 * _normal((case["m"], case["nh"] * case["hd"]), _gen(seed, 1))
    return q, _normal((rows, kvd), _gen(seed, 2)).half(), _normal((rows, kvd), _gen(seed, 3)).half()


def _logits(case, seed):
    return 2.5 * _normal((case["n"],), _gen(seed, 1))


def prepare(case, seed):
    mxhip.init(0)
    op = case["op"]
    s = {"case": case}
    if op == "model":
        path = _model_file(case, seed)
        s["model"] = mxhip.Model(path, case["n_ctx"])
        os.unlink(path)
        s["prompt"], s["ids"] = _model_ids(case, seed)
    elif op in ("gemv", "rows", "gemm"):
        s["w"], s["x"] = _matvec_inputs(case, seed)
        s["type"] = TYPES[case["type"]]
        torch.cuda.synchronize()
        if case.get("tiled"):
            for w in s["w"]:
                t = ctypes.c_int(-1)
                mxhip.check(mxhip.lib.mxh_tile_rows(TYPES[case["type"]], w.data_ptr(), case["n"], case["k"],
                                                    ctypes.byref(t)), "mxh_tile_rows")
                s["type"] = t.value
        s["y"] = torch.empty((case.get("count", 1), case.get("m", 1), case["n"]), device="cuda")
    elif op == "attention":
        s["q"], s["k"], s["v"] = _attention_inputs(case, seed)
        s["att"] = torch.empty_like(s["q"])
    elif op == "dequant":
        s["w"] = _raw(case["type"], case["rows"], case["cols"], seed, 10)
        s["out"] = torch.empty((case["rows"], case["cols"]), device="cuda")
    else:
        s["logits"], s["seed"] = _logits(case, seed), seed
        # a resident handle that mxhip.sample takes
        s["buf"] = mxhip.DeviceBuffer.from_array(s["logits"].cpu().numpy())
    mxhip.synchronize()
    torch.cuda.synchronize()
    return s


def run(s):
    c, op = s["case"], s["case"]["op"]
    if op == "model":
        m = s["model"]
        m.reset()
        m.prefill(s["prompt"])
        return np.stack([m.step(int(t))[0] for t in s["ids"]])
    if op == "gemv":
        x, y, n = s["x"].data_ptr(), s["y"].data_ptr(), c["n"]
        for i, w in enumerate(s["w"]):
            mxhip.gemv(s["type"], w.data_ptr(), x, y + 4 * i * n, n, c["k"], c["form"])
        return s["y"]
    if op in ("rows", "gemm"):
        f = mxhip.lib.mxh_matmul_rhs_t if op == "rows" else mxhip.lib.mxh_gemm_q_f16
        mxhip.check(f(s["type"], s["x"].data_ptr(), c["m"], s["w"][0].data_ptr(), c["n"], c["k"], s["y"].data_ptr(),
                      c["form"]), op)
        return s["y"]
    if op == "attention":
        mxhip.check(mxhip.lib.mxh_attention_prefill(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                                    s["att"].data_ptr(), c["p0"], c["m"], c["nh"], c["nkv"], c["hd"]),
                    op)
        return s["att"]
    if op == "dequant":
        mxhip.check(mxhip.lib.mxh_dequant(TYPES[c["type"]], s["w"].data_ptr(), s["out"].data_ptr(), c["rows"],
                                          c["cols"], c["form"]), op)
        return s["out"]
    return mxhip.sample(s["buf"], c["n"], c["top_k"], c["temperature"], c["top_p"], c["min_p"], s["seed"], 3)


def work(case):
    op = case["op"]
    if op == "model":
        a, t, n = ARCHS[case["arch"]], case["prompt"], case["steps"]
        types = [TYPES[x] for x in MIXES[case["mix"]]]
        qd, kvd, d, f, layers = (a["n_head"] * a["head_dim"], a["n_head_kv"] * a["head_dim"], a["n_embd"], a["n_ff"],
                                 case["layers"])
        # (type, rows, cols) of a layer's matrices
        mats = [(types[0], qd + kvd, d), (types[1], kvd, d), (types[0], d, qd), (types[0], 2 * f, d), (types[1], d, f)]
        layer = sum(r * mxhip.row_bytes(ty, c) for ty, r, c in mats)
        head = a["n_vocab"] * mxhip.row_bytes(types[2], d)
        # the weights once for the prompt and once per step, the K/V rows of every step, the logits out
        kv = sum(4 * kvd * (t + i) for i in range(n)) * layers
        lin = 2 * sum(r * c for _, r, c in mats) * layers
        att = 4 * qd * sum(range(1, t + n + 1)) * layers
        return {"bytes": layers * layer * (1 + n) + n * (head + 4 * a["n_vocab"]) + kv,
                "flops": lin * (t + n) + att + 2 * n * a["n_vocab"] * d}
    if op in ("gemv", "rows", "gemm"):
        m, n, k, count = case.get("m", 1), case["n"], case["k"], case.get("count", 1)
        return {"bytes": count * (n * mxhip.row_bytes(TYPES[case["type"]], k) + 4 * m * n) + 4 * m * k,
                "flops": 2 * count * m * n * k}
    if op == "attention":
        m, p0, qd, kvd = case["m"], case["p0"], case["nh"] * case["hd"], case["nkv"] * case["hd"]
        return {"bytes": 8 * m * qd + 4 * (p0 + m) * kvd, "flops": 4 * qd * (m * p0 + m * (m + 1) // 2)}
    if op == "dequant":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * mxhip.row_bytes(TYPES[case["type"]], c) + 4 * r * c, "flops": 2 * r * c}
    return {"bytes": 4 * case["n"], "flops": case["n"]}


def tolerance(case):
    """About four times the distance to the 64-bit results that the paths show over these ranges."""
    op = case["op"]
    if op in ("dequant", "sample"):  # bit-exact decoding; one id
        return "exact"
    if op == "model":  # 1e-5 .. 1.2e-4: fp32 roundings amplified by fp16 rounding flips of cache entries
        return {"rel": 6e-4}
    if op == "attention":  # 1e-5: probabilities as a pair of fp16
        return {"rel": 5e-5}
    return {"rel": 2e-6}  # 1e-7 .. 5e-7: fp32 sums


# ---- 64-bit references -----------------------------------------------------------------


def _product(x, raw, name, form):
    """x . decode(raw)^T in float64, a slab of weight rows at a time."""
    x = x.double()
    step = max(1, (1 << 26) // x.shape[-1])
    return torch.cat([x @ decode(raw[r:r + step], name, form).T for r in range(0, raw.shape[0], step)], -1)


def _read_gguf(path):
    """name -> (type id, rows, cols, raw uint8 rows) of a GGUF v3 file's tensors."""
    data = np.memmap(path, np.uint8, "r")
    at = 8
    fixed = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, data, at)
        at += struct.calcsize("<" + fmt)
        return v if len(v) > 1 else v[0]

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(data[at - n:at]).decode()

    def skip(kind):
        nonlocal at
        if kind == 8:
            text()
        elif kind == 9:
            inner, n = take("IQ")
            for _ in range(n):
                skip(inner)
        else:
            at += fixed[kind]

    n_tensors, n_kv = take("QQ")
    align = 32
    for _ in range(n_kv):
        key, kind = text(), take("I")
        if key == "general.alignment":
            align = struct.unpack_from("<I", data, at)[0]
        skip(kind)
    entries = []
    for _ in range(n_tensors):
        name, dims = text(), take("I")
        ne = [take("Q") for _ in range(dims)]
        kind, off = take("IQ")
        entries.append((name, kind, ne[1] if dims > 1 else 1, ne[0], off))
    base = (at + align - 1) // align * align
    names = {v: k for k, v in TYPES.items()}
    out = {}
    for name, kind, rows, cols, off in entries:
        width = mxhip.row_bytes(kind, cols)
        out[name] = (names[kind], np.array(data[base + off:base + off + rows * width]).reshape(rows, width))
    return out


def _exact_model(case, seed):
    path = _model_file(case, seed)
    t = _read_gguf(path)
    os.unlink(path)
    a = ARCHS[case["arch"]]
    nh, nkv, hd = a["n_head"], a["n_head_kv"], a["head_dim"]

    def w(name):
        kind, raw = t[name]
        return kind, torch.from_numpy(raw).cuda()

    def vec(name):
        return decode(w(name)[1], "F32")[0]

    def proj(x, name):
        kind, raw = w(name)
        return _product(x, raw, kind, 0)

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + a["eps"]) * g

    prompt, ids = _model_ids(case, seed)
    seq = torch.from_numpy(np.concatenate([prompt, ids])).long()
    n = len(seq)
    kind, raw = t["token_embd.weight"]
    x = decode(torch.from_numpy(raw[seq.numpy()]).cuda(), kind)
    ang = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * \
        (a["rope_theta"] ** (-torch.arange(0, hd, 2, dtype=torch.float64, device="cuda") / hd))
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(v):  # adjacent pairs
        p, q = v[..., 0::2], v[..., 1::2]
        return torch.stack([p * cos - q * sin, p * sin + q * cos], -1).flatten(-2)

    mask = torch.full((n, n), -math.inf, dtype=torch.float64, device="cuda").triu(1)
    for i in range(case["layers"]):
        p = "blk.%d." % i
        h = norm(x, vec(p + "attn_norm.weight"))
        q, k, v = (proj(h, p + "attn_%s.weight" % c).reshape(n, -1, hd) for c in "qkv")
        if a["qk_norm"]:
            q, k = norm(q, vec(p + "attn_q_norm.weight")), norm(k, vec(p + "attn_k_norm.weight"))
        q, k, v = rope(q), rope(k).half().double(), v.half().double()  # the cache is fp16
        heads = [torch.softmax(q[:, j] @ k[:, j * nkv // nh].T / math.sqrt(hd) + mask, -1) @ v[:, j * nkv // nh]
                 for j in range(nh)]
        x = x + proj(torch.cat(heads, -1), p + "attn_output.weight")
        h = norm(x, vec(p + "ffn_norm.weight"))
        g = proj(h, p + "ffn_gate.weight")
        x = x + proj(g * torch.sigmoid(g) * proj(h, p + "ffn_up.weight"), p + "ffn_down.weight")
    h = norm(x[len(prompt):], vec("output_norm.weight"))
    return proj(h, "token_embd.weight" if a["tied"] else "output.weight").cpu().numpy()


def _exact_sample(case, seed):
    """top-k by (logit, lower id), softmax at T, top-p and min-p cuts, a splitmix64 draw."""
    lg = _logits(case, seed).cpu().numpy()
    order = np.lexsort((np.arange(lg.size), -lg.astype(np.float64)))[:case["top_k"]]
    p = np.exp((lg[order].astype(np.float64) - float(lg[order[0]])) / case["temperature"])
    p /= p.sum()
    if case["top_p"] < 1:
        p = p[:int(np.searchsorted(np.cumsum(p), case["top_p"])) + 1]
        p /= p.sum()
    if case["min_p"] > 0:
        p = p[p >= p[0] * case["min_p"]]
        p /= p.sum()
    z = (seed + 4 * 0x9E3779B97F4A7C15) & (2**64 - 1)
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & (2**64 - 1)
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & (2**64 - 1)
    u = ((z ^ (z >> 31)) >> 11) / 2.0**53 * p.sum()
    return int(order[min(int(np.searchsorted(np.cumsum(p), u, side="right")), len(p) - 1)])


def exact(case, seed):
    op = case["op"]
    if op == "model":
        return _exact_model(case, seed)
    if op in ("gemv", "rows", "gemm"):
        ws, x = _matvec_inputs(case, seed)
        return torch.stack([_product(x, w, case["type"], case["form"]) for w in ws])
    if op == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        m, p0, nh, nkv, hd = (case[x] for x in ("m", "p0", "nh", "nkv", "hd"))
        hidden = torch.arange(p0 + m, device="cuda")[None] > p0 + torch.arange(m, device="cuda")[:, None]
        out = []
        for h in range(nh):
            g = h * nkv // nh
            s = q[:, h * hd:(h + 1) * hd] @ k[:, g * hd:(g + 1) * hd].T / math.sqrt(hd)
            out.append(torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, g * hd:(g + 1) * hd])
        return torch.cat(out, -1)
    if op == "dequant":
        return decode(_raw(case["type"], case["rows"], case["cols"], seed, 10), case["type"], case["form"])
    return _exact_sample(case, seed)
