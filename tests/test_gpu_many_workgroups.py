"""The device-decided step of many workgroups in one launch: ragged, short, empty and unaligned chunks up to the end of its range.  That these lists
are done so is checked in test_scratch_routes.py."""
import pytest
import torch

import test_gpu_step_scratch as scratch
from patrickstar_amd import _lib, adam_op
from test_gpu_short_lists import OPT

pytestmark = pytest.mark.gpu
MOST = 280 * 256  # elements of the longest list that is one launch

# chunks, chunk length, used lengths (None: all full), element offset of the payloads in their allocations
LISTS = [
    (1, MOST, None, 0), (1, MOST, [MOST - 100], 3), (3, 16 * 256 + 1, None, 0), (7, 40 * 256 - 3, [40 * 256 - 3, 10000, 256, 255, 1, 0, 40 * 256 - 3], 0),
    (64, 1000, None, 4), (2, 35000, [34999, 3], 1), (5, 56 * 256, [56 * 256, 1, 0, 4097, 4095], 2), (40, 7 * 256, [1792, 1, 256, 0] * 10, 0),
]


@pytest.mark.parametrize("case", LISTS, ids=[f"{c[0]}x{c[1]}at{c[3]}" for c in LISTS])
@pytest.mark.parametrize("arithmetic,adamw,wd,clamp,scale,eps", [
    (0, True, 0.01, 0.0, 2.0**12, 1e-8), (0, False, 0.01, 1.0, 1000.0, 1e-8), (1, True, 0.0, 0.0, 2**16, 1e-8), (0, True, 0.01, 0.0, 2.0**12, 0.0),
])
def test_one_launch_is_its_three_parts(case, arithmetic, adamw, wd, clamp, scale, eps):
    scratch.test_one_launch_is_its_three_parts(case, arithmetic, adamw, wd, clamp, scale, eps)


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
