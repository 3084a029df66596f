"""Updates whose workgroups all fit the GPU at once are launched without the request that caps the resident ones: both sides of that
line, in each form that has it, against the oracle, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
LINE = 8192 * 256  # elements that are resident at once
OPT = 8301
HYPER = (1e-3, 0.9, 0.999, 1e-8, 0.01)
SCALE = 2.0**12


def _lists(n):
    rng = np.random.default_rng(n)
    p, m = ((rng.standard_normal(n) * f).astype(np.float32) for f in (0.02, 1e-4))
    return p, m, (rng.standard_normal(n) * 1e-4).astype(np.float32) ** 2, (rng.standard_normal(n) * 1e-3 * SCALE).astype(np.float16)


@pytest.mark.parametrize("form", ["chunk", "descriptors", "device", "tensors", "each", "operator"])
@pytest.mark.parametrize("n", [LINE - 257, LINE - 1, LINE, LINE + 1])
def test_both_sides_of_the_line(form, n):
    lib, s = _lib.load(), _lib.current_stream_handle()
    p, m, v, g = _lists(n)
    lists = [torch.from_numpy(x).cuda() for x in (p, m, v, g)]
    rows = lambda *at: _lib.chunk_array([[t[a:].data_ptr() for t in lists] for a in at])  # noqa: E731
    cut = n // 3 // 256 * 256 + (5 if form == "descriptors" else 0)
    numels = (ctypes.c_size_t * 2)(cut, n - cut)
    steps = (1, 2)
    adam_op.create_adam(OPT, *HYPER, True, False)
    scaler = DynamicLossScaler(init_scale=SCALE).materialize("cuda:0", betas=HYPER[1:3]) if form == "device" else None
    out = torch.zeros(n, dtype=torch.half, device="cuda")
    for step in steps:
        lists[3].copy_(torch.from_numpy(g))
        if form == "chunk":
            rc = lib.ps_adam_step_chunks(OPT, step, *HYPER, 1, rows(0), 1, n, None, None, SCALE, s)
        elif form == "descriptors":
            rc = lib.ps_adam_step_chunks(OPT, step, *HYPER, 1, rows(0, cut), 2, n - cut, numels, None, SCALE, s)
        elif form == "device":
            rc = lib.ps_adam_step_chunks_dynamic_scratch(OPT, HYPER[0], *HYPER[3:], 1, rows(0), 1, n, None, None, 1, scaler.state_ptr, None, 0, 1,
                                                         scaler._scratch.data_ptr(), _lib.PS_STEP_SCRATCH_BYTES, s)
        elif form == "tensors":
            rc = lib.ps_adam_step_tensors(OPT, step, *HYPER, 1, rows(0, cut), numels, 2, None, SCALE, None, s)
        elif form == "each":
            calls = (_lib.ps_tensor_call * 2)(*[(*HYPER, step, -1, 0)] * 2)
            rc = lib.ps_adam_step_tensors_each(OPT, 1, rows(0, cut), numels, calls, 2, SCALE, None, None, 0, s)
        else:
            rc = lib.ps_adam_update(OPT, step, *HYPER, 1, lists[0].data_ptr(), lists[3].data_ptr(), 1, lists[1].data_ptr(), lists[2].data_ptr(), n,
                                    SCALE, out.data_ptr(), s)
        _lib.check(rc, form)
    adam_op.destroy_adam(OPT)
    ref = oracle.AdamOracle(*HYPER, True)
    for step in steps:
        ref.update(step, *HYPER, True, p, g, m, v, SCALE)
    got = [t.cpu().numpy() for t in (*lists[:3], out if form == "operator" else lists[3])]
    for what, a, b in zip(("p", "m", "v", "h"), got, (p, m, v, oracle.cast_fp32_to_fp16(p))):
        a, b = (x.reshape(-1).view(np.uint8) for x in (a, b))
        assert np.array_equal(a, b), what
