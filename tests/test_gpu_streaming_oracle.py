"""Tensor lists that stream past the caches, next to the CPU oracle (chunk lists of that length: test_gpu_adam_parity.py)."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from patrickstar_amd import _lib, adam_op
from _harness import assert_bits_equal

pytestmark = pytest.mark.gpu
MI = 1 << 20
OPT = 8301
SIZES = [16 * MI, 3, 12 * MI + 1, 255, 1 * MI, 500_000]
LR, B1, B2, EPS, WD, SCALE = 1e-3, 0.9, 0.999, 1e-8, 0.01, 2.0**12


@pytest.mark.parametrize("each", [False, True])
@pytest.mark.parametrize("packed", [True, False])  # at one distance, one launch; the last variance further on: several
def test_tensor_lists_next_to_the_oracle(packed, each):
    total, scale = sum(SIZES) + 1024, SCALE
    rng = np.random.default_rng(7)
    host = {k: rng.standard_normal(total, dtype=np.float32) * np.float32(f) for k, f in (("p", 0.02), ("m", 1e-4), ("v", 1e-3), ("h", 1e-3 * scale))}
    host["v"], host["h"] = np.square(host["v"]), host["h"].astype(np.float16)
    dev = {k: torch.from_numpy(a.copy()).cuda() for k, a in host.items()}
    at = np.cumsum([0] + SIZES)[:-1]
    at_v = at if packed else np.append(at[:-1], at[-1] + 1024)
    rows = _lib.chunk_array([[dev["p"][a:].data_ptr(), dev["m"][a:].data_ptr(), dev["v"][b:].data_ptr(), dev["h"][a:].data_ptr()] for a, b in zip(at, at_v)])
    numels, n = (ctypes.c_size_t * len(SIZES))(*SIZES), len(SIZES)
    lib, s = _lib.load(), _lib.current_stream_handle()
    adam_op.create_adam(OPT, LR, B1, B2, EPS, WD, True, False)
    if each:
        calls = (_lib.ps_tensor_call * n)(*[(LR * (i + 1), B1, B2, EPS, WD, 3, -1, 0) for i in range(n)])
        rc = lib.ps_adam_step_tensors_each(OPT, 1, rows, numels, calls, n, scale, None, None, 0, s)
    else:
        rc = lib.ps_adam_step_tensors(OPT, 3, LR, B1, B2, EPS, WD, 1, rows, numels, n, None, scale, None, s)
    _lib.check(rc, "step")
    adam_op.destroy_adam(OPT)
    native = oracle.AdamOracle(LR, B1, B2, EPS, WD, True)
    for i, (a, b, k) in enumerate(zip(at, at_v, SIZES)):
        p, h, m, v = host["p"][a:][:k], host["h"][a:][:k], host["m"][a:][:k], host["v"][b:][:k]
        native.update(3, LR * (i + 1) if each else LR, B1, B2, EPS, WD, True, p, h, m, v, scale)
        h[...] = oracle.cast_fp32_to_fp16(np.ascontiguousarray(p))
    for k in "pmvh":
        assert_bits_equal(dev[k].cpu().numpy(), host[k], k)
