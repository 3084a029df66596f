"""The device-decided step of many workgroups in one launch: ragged, short, empty and unaligned chunks up to the end of its range, and
the marks that workgroups leave one another in the scratch memory, as a workgroup that starts late finds them.  That these lists
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


DIRTY, CLEAN, TICKETS = 192 // 8, 200 // 8, 128 // 4  # words of StepScratch (csrc/ps_kernels.h); the first one counts launches
# what the gradients say, mark, how far it is from the launches so far (1: of this launch), whether the step is to be skipped
MARKS = [(False, DIRTY, 1, True), (True, CLEAN, 1, False), (False, DIRTY, 0, False), (True, CLEAN, 0, True), (True, DIRTY, 1, True),
         (False, CLEAN, 1, False), (True, DIRTY, 0, True), (False, CLEAN, 0, False)]


@pytest.mark.parametrize("case", [(3, 9 * 256 + 5, None, 0), (5, 50 * 256, [12800, 1, 0, 4097, 4095], 1)], ids=["even", "ragged"])
@pytest.mark.parametrize("launches", [0, 7, 2**32 - 2, 2**32 - 1])
def test_a_mark_of_the_launch_decides_and_an_old_one_does_not(case, launches):
    """A mark that was there before a workgroup's look is what a late start comes to: others have replaced gradients, and the mark says
    whether by parameters of a clean step or of a skipped one.  (The clamp keeps the update by an infinity finite.)"""
    a, b = [scratch._Scratched(one, case, 0, False, 0.01, 1.0, 1000.0, 1e-8) for one in (False, True)]
    words, counts = b.scaler._scratch.view(torch.int64), b.scaler._scratch.view(torch.int32)
    n_chunks, n, used, offset = case
    sizes = [n] * n_chunks if used is None else used
    flag = _lib.ps_step_state.overflow.offset
    for k, (infinite, mark, age, skip) in enumerate(MARKS):
        for r in (a, b):
            for i, size in enumerate(sizes):
                r.lists[3][i, offset : offset + size] = (r.lists[0][i, offset : offset + size] * 50).half()
            if infinite:
                r.lists[3][n_chunks - 1, offset + sizes[-1] - 1] = float("inf")
        words.zero_()
        words[0] = launches
        words[mark] = launches + age
        b.step(1, 3, (0, 0, 100))
        if skip:  # the parts are told by the flag, without a probe
            a.scaler._state[flag : flag + 4].view(torch.int32).fill_(1)
        a.step(0, 3, (0, 0, 100))
        for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a.lists, b.lists):
            kind = torch.int16 if x.dtype == torch.half else torch.int32
            assert torch.equal(x.view(kind), y.view(kind)), (k, name)
        assert torch.equal(a.scaler._state, b.scaler._state) and torch.equal(a.scaler._log, b.scaler._log), k
        assert b.scaler.last_step_skipped == skip, k
        assert words[0] == launches + 1 and counts[TICKETS] == 0, k
    for one in (0, 1):
        adam_op.destroy_adam(OPT + one)


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
