"""The device-decided step by many workgroups in one launch (with scratch memory), against the probe, the step and the scale update
as calls of their own: payloads, step state and log the same bits.  Lists around the ends of a workgroup's tiles and of the range,
ragged and unaligned ones, overflows in any tile, steps whose parameters do not fit binary16 (a workgroup that starts late then finds
infinities where others found gradients), and clean steps behind each of them, which old marks must not reach."""
import pytest
import torch

from patrickstar_amd import _lib, adam_op
from test_gpu_short_lists import OPT, _Run

pytestmark = pytest.mark.gpu
SPAN = 15 * 256  # elements of the tiles a workgroup has in hand
MOST = 400 * 256

LISTS = [
    (1, 1, None, 0), (1, SPAN, None, 0), (1, SPAN + 1, None, 0), (3, 6267, None, 0), (1, 16 * SPAN + 255, None, 0), (1, MOST, None, 0), (1, MOST + 1, None, 0),
    (7, 14501, [14501, 14000, 256, 255, 1, 0, 14501], 0), (64, 1500, None, 4), (65, 1250, None, 0), (2, 50000, [49999, 3], 1), (24, 9 * 256, None, 0),
]


class _Scratched(_Run):
    def step(self, probe, operator_calls, span):
        if not self.one_call:
            return super().step(probe, operator_calls, span)
        n_chunks, n, used, _ = self.case
        calls = _lib.call_pattern(operator_calls, *span) if operator_calls else None
        scratch = self.scaler._scratch
        _lib.check(_lib.load().ps_adam_step_chunks_dynamic_scratch(
            OPT + 1, 1e-3, self.eps, self.wd, 1, self.table, n_chunks, n, self.used, calls, int(probe), self.scaler.state_ptr,
            *self.scaler.log_arguments(), operator_calls, scratch.data_ptr(), scratch.numel(), _lib.current_stream_handle()), "one launch")


@pytest.mark.parametrize("case", LISTS, ids=[f"{c[0]}x{c[1]}" for c in LISTS])
@pytest.mark.parametrize("arithmetic,adamw,wd,clamp,scale,eps", [
    (0, True, 0.01, 0.0, 2.0**12, 1e-8), (0, False, 0.01, 1.0, 1000.0, 1e-8), (1, True, 0.0, 0.0, 2**16, 1e-8), (0, True, 0.01, 0.0, 2.0**12, 0.0),
])
def test_one_launch_is_its_three_parts(case, arithmetic, adamw, wd, clamp, scale, eps):
    runs = [_Scratched(one, case, arithmetic, adamw, wd, clamp, scale, eps) for one in (False, True)]
    n_chunks, n, used, offset = case
    sizes = [n] * n_chunks if used is None else used
    last = max(i for i in range(n_chunks) if sizes[i])
    span = (last, 0, sizes[last] // 2)
    gen = torch.Generator().manual_seed(n)
    # (what goes in, probe, flag raised before)
    steps = [("", 1, 0), ("inf", 1, 0), ("large", 1, 0), ("nan", 1, 0), ("", 0, 1), ("large", 1, 1), ("", 0, 0), ("all", 1, 0), ("", 1, 0), ("large", 0, 0), ("inf", 1, 0), ("", 1, 0)]
    for k, (what, probe, flag) in enumerate(steps):
        bad = [(i, int(torch.randint(sizes[i], (1,), generator=gen))) for i in range(n_chunks) if sizes[i]]
        place = [bad[0], bad[-1], (last, sizes[last] - 1)][k % 3]
        for r in runs:
            grads, masters = r.lists[3], r.lists[0]
            grads[:, offset : offset + n] = torch.where(masters[:, offset : offset + n] == 0, 0.0, grads[:, offset : offset + n].nan_to_num(1, 1, 1).clamp(-9, 9) * 50).half()
            if what in ("inf", "nan"):
                grads[place[0], offset + place[1]] = float(what)
            if what == "all":
                grads[:, offset : offset + 1 + n // 3] = float("nan")
            for i, at in bad if what == "large" else ():
                masters[i, offset + at] = 1e6  # an infinity as binary16
            if flag:
                r.scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            r.step(probe, 0 if arithmetic else (1 if k == 3 else 3), (0, 0, 0) if k == 3 else span)
        a, b = runs
        for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a.lists, b.lists):
            kind = torch.int16 if x.dtype == torch.half else torch.int32
            assert torch.equal(x.view(kind), y.view(kind)), (k, what, name)
        assert torch.equal(a.scaler._state, b.scaler._state), (k, what)
        assert a.scaler.last_step_skipped == (what in ("inf", "nan", "all") or bool(flag))
        assert torch.equal(a.scaler._log, b.scaler._log), (k, what)
    for one in (0, 1):
        adam_op.destroy_adam(OPT + one)


def test_scratch_that_is_too_small_or_unaligned_is_refused():
    r = _Scratched(1, (1, 300, None, 0), 0, True, 0.01, 0.0, 2.0**12, 1e-8)
    f, state, s = _lib.load().ps_adam_step_chunks_dynamic_scratch, r.scaler.state_ptr, _lib.current_stream_handle()
    at = r.scaler._scratch.data_ptr()
    for place, size in ((at, 255), (at + 32, 256)):
        assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, None, 0, 1, place, size, s) == _lib.PS_ERR_BAD_ARG
    adam_op.destroy_adam(OPT + 1)
