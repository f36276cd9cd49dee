"""Device memory the batched prefill takes per model (GPU): the chunk buffers,
and no split-K buffer of its own (that is the library stream's).
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import mxhip

pytestmark = pytest.mark.gpu


def free_bytes():
    hip, free, total = C.CDLL("libamdhip64.so.7"), C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("wtype,flags", [(mxhip.Q4_K, 0), (mxhip.Q4_K, mxhip.MODEL_BF16_PREFILL)], ids=["codes", "bf16"])
def test_prefill_allocates_its_chunk_buffers_only(mxh, tmp_path, wtype, flags):
    d, nh, nkv, hd, f, rows = 4096, 32, 8, 128, 4096, 512
    path = tmp_path / "m.gguf"
    mxhip.write_synthetic_gguf(path, n_layer=1, n_embd=d, n_head=nh, n_head_kv=nkv, head_dim=hd, n_ff=f, n_vocab=512,
                               ctx=1024, wtype=wtype)
    m = mxhip.Model(path, 640, flags)
    before = free_bytes()
    m.prefill(np.zeros(520, np.int32))
    took = before - free_bytes()
    qd, kvd = nh * hd, nkv * hd
    # fp32 x, q|k|v, q, attention, gate|up; the GEMM inputs as two bf16 and two
    # fp16 arrays; up to 2 MiB of rounding for each of the 12 allocations.  (A
    # buffer for four splits of q|k|v would be 48 MiB more.)
    need = rows * (4 * (d + qd + 2 * kvd + 2 * qd + 2 * f) + 4 * 2 * max(d, f))
    assert took <= need + 12 * (2 << 20), f"{took / 2**20:.0f} MiB for {need / 2**20:.0f}"
    del m
