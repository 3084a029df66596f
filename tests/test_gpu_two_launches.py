"""The device-decided step in two launches (probe and copy of the state; update and scale update), against the probe, the step and the
scale update as calls of their own: payloads, step state and log the same bits.  Evenly spaced lists, lists with descriptors
(unaligned, ragged, unevenly spaced), both sides of the lines, overflows on steps next to one another (the probe has a word for every other step,
which the step between must have cleared), steps without a probe in between."""
import pytest
import torch

from patrickstar_amd import _lib, adam_op
from test_gpu_short_lists import OPT
from test_gpu_step_scratch import _Scratched

pytestmark = pytest.mark.gpu
ONE = 280 * 256  # elements of the longest list that is one launch
PROBE = 64 * 8 * 8  # elements that a wave probes

LISTS = [
    (1, ONE, None, 0), (1, ONE + 1, None, 0), (5, 4 * PROBE, None, 0), (5, 4 * PROBE + 1, [4 * PROBE + 1] * 4 + [1], 0), (1, 3 << 19, None, 0),
    (7, 20501, [20501, 14000, 256, 255, 1, 0, 20501], 0), (64, 2500, None, 4), (65, 2304, None, 0), (2, 100003, [99999, 3], 1),
    (2, (16 << 20) + 8, None, 0), (2, (16 << 20) + 3, None, 0),
]


@pytest.mark.parametrize("case", LISTS, ids=[f"{c[0]}x{c[1]}" for c in LISTS])
@pytest.mark.parametrize("arithmetic,adamw,wd,clamp,scale,eps", [
    (0, True, 0.01, 0.0, 2.0**12, 1e-8), (0, False, 0.01, 1.0, 1000.0, 1e-8), (1, True, 0.0, 0.0, 2**16, 1e-8), (0, True, 0.01, 0.0, 2.0**12, 0.0),
])
def test_two_launches_are_their_three_parts(case, arithmetic, adamw, wd, clamp, scale, eps):
    runs = [_Scratched(one, case, arithmetic, adamw, wd, clamp, scale, eps) for one in (False, True)]
    n_chunks, n, used, offset = case
    sizes = [n] * n_chunks if used is None else used
    last = max(i for i in range(n_chunks) if sizes[i])
    span = (last, 0, sizes[last] // 2)
    first, end = (0, 0), (last, sizes[last] - 1)
    # (overflow, where, probe, flag raised before)
    steps = [(0, first, 1, 0), (1, end, 1, 0), (1, first, 1, 0), (0, first, 1, 0), (1, end, 1, 1), (0, first, 1, 0), (0, first, 0, 1), (1, end, 1, 0),
             (0, first, 0, 0), (0, first, 1, 1), (0, first, 1, 0), (0, first, 1, 0)]
    for k, (poison, place, probe, flag) in enumerate(steps):
        for r in runs:
            grads, masters = r.lists[3], r.lists[0]
            grads[:, offset : offset + n] = torch.where(masters[:, offset : offset + n] == 0, 0.0, grads[:, offset : offset + n].nan_to_num(1, 1, 1).clamp(-9, 9) * 50).half()
            if poison:
                grads[place[0], offset + place[1]] = float("nan") if k % 2 else float("inf")
            if flag:
                r.scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            r.step(probe, 0 if arithmetic else (1 if k == 3 else 3), (0, 0, 0) if k == 3 else span)
        a, b = runs
        for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a.lists, b.lists):
            kind = torch.int16 if x.dtype == torch.half else torch.int32
            assert torch.equal(x.view(kind), y.view(kind)), (k, name)
        assert torch.equal(a.scaler._state, b.scaler._state), k
        assert a.scaler.last_step_skipped == bool(poison or flag)
        assert torch.equal(a.scaler._log, b.scaler._log), k
    for one in (0, 1):
        adam_op.destroy_adam(OPT + one)


def test_a_captured_step_in_two_launches_replays_as_it_ran():
    """Replays with steps outside the graph and an overflow in between: the scratch carries which word the next probe writes."""
    case = (3, 100003, None, 0)
    runs = [_Scratched(one, case, 0, True, 0.01, 0.0, 2.0**12, 1e-8) for one in (False, True)]
    a, b = runs
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for r in runs:
            r.step(1, 3, (0, 0, 100))
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            b.step(1, 3, (0, 0, 100))
        for k in range(7):
            for r in runs:
                r.lists[3].copy_((r.lists[0] * 50).half())
                if k in (1, 2, 4):
                    r.lists[3][k % 3, 100002] = float("inf")
            a.step(1, 3, (0, 0, 100))
            if k == 3:
                b.step(1, 3, (0, 0, 100))
            else:
                graph.replay()
            stream.synchronize()
            assert all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(a.lists, b.lists)), k
            assert torch.equal(a.scaler._state, b.scaler._state), k
            assert a.scaler.last_step_skipped == (k in (1, 2, 4))
    for one in (0, 1):
        adam_op.destroy_adam(OPT + one)
