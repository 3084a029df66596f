"""The scratch memory of device-decided steps."""
import pytest
import torch

import test_gpu_step_scratch as scratch
from patrickstar_amd import _lib, adam_op
from test_gpu_short_lists import OPT

pytestmark = pytest.mark.gpu


def test_scratch_one_byte_short_or_off_its_line_is_refused():
    r = scratch._Scratched(1, (1, 300, None, 0), 0, True, 0.01, 0.0, 2.0**12, 1e-8)
    f, state, s = _lib.load().ps_adam_step_chunks_dynamic_scratch, r.scaler.state_ptr, _lib.current_stream_handle()
    memory = torch.zeros(_lib.PS_STEP_SCRATCH_BYTES + 64, dtype=torch.uint8, device="cuda")
    at, whole = memory.data_ptr(), _lib.PS_STEP_SCRATCH_BYTES
    for place, size in ((at, whole - 1), (at + 32, whole), (at + 8, whole), (at + 1, whole)):
        assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, None, 0, 1, place, size, s) == _lib.PS_ERR_BAD_ARG
    assert r.scaler.cur_iter == 0
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, None, 0, 1, at, whole, s) == 0
    assert r.scaler.cur_iter == 1
    adam_op.destroy_adam(OPT + 1)
