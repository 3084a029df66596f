"""Tensors that lie at the same place of their four lists take one launch of the one-dimensional kernels; any other list takes the
two-dimensional ones.  Both are run over the same numbers (for the second, one tensor's variance lies one element further on)
and have to leave the same bits, whatever the lengths, phases, order and number of the tensors, the step's decision and its classes."""
import ctypes
import random

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
T = 256  # elements per tile
OPT = 7701

SHAPES = {
    "one": [5 * T + 3],
    "equal_lengths": [33 * T] * 40,
    "short": [1, 2, 3, 255, 256, 257, 768] * 12,
    "ends_of_segments": [31 * T, 32 * T, 32 * T + 1, 33 * T, 34 * T, 36 * T, 37 * T, 40 * T - 1, 1000 * T, 900 * T, 899 * T, 1],
    "ten_segments": [int(40 * T * 1.3**k) + k for k in range(10)] + [7] * 5,
    "three_launches": [64 + 5 * k for k in range(209)] + [300] * 208 + [40 * T],
    "with_empty": [0, 700, 0, 33 * T + 1, 0],
    "layer": ([768 * T] + [3 * T] * 4 + [2304 * 4 * T, 12 * T]) * 3,
}


class Lists:
    def __init__(self, sizes, gap, moved, scale, seed):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        order = list(range(len(sizes)))
        random.Random(seed).shuffle(order)
        at, cursor = [0] * len(sizes), 5 if gap else 0
        for i in order:
            at[i] = cursor
            cursor += sizes[i] + gap
        n = cursor + 64
        self.data = [torch.randn(n, device="cuda", generator=gen) * f for f in (0.02, 1e-4, 1e-3)]
        self.data[2].square_()
        self.data.append((torch.randn(n, device="cuda", generator=gen) * 1e-3 * scale).clamp_(-6e4, 6e4).half())
        rows = [[t[a:].data_ptr() for t in self.data] for a in at]
        self.own = None
        if moved:  # the last tensor's variance: a copy, one element off its phase
            k = max(range(len(sizes)), key=lambda i: (sizes[i] > 0, i))
            self.own = torch.empty(sizes[k] + 1, device="cuda")
            self.own[1:] = self.data[2][at[k] : at[k] + sizes[k]]
            self.back = self.data[2][at[k] : at[k] + sizes[k]]
            rows[k][2] = self.own[1:].data_ptr()
        self.rows, self.numels, self.n = _lib.chunk_array(rows), (ctypes.c_size_t * len(sizes))(*sizes), len(sizes)

    def whole(self):
        if self.own is not None:
            self.back.copy_(self.own[1:])
        return self.data


def _run(sizes, gap, moved, decided, classes, arithmetic, scale):
    lib, s = _lib.load(), _lib.current_stream_handle()
    lists = Lists(sizes, gap, moved, scale, seed=len(sizes) + gap)
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    lib.ps_adam_set_arithmetic(OPT, arithmetic)
    scaler = None
    if decided != "host":
        scaler = DynamicLossScaler(init_scale=scale).materialize("cuda:0", betas=(0.9, 0.999))
        if decided == "skipped":
            scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
    state = scaler.state_ptr if scaler is not None else None
    for step in (1, 2):
        if classes:
            each = (_lib.ps_tensor_call * lists.n)()
            for i in range(lists.n):
                d = step if scaler is None else 0
                each[i] = _lib.ps_tensor_call(1e-3 * 0.9 ** (i % classes), 0.9, 0.999, 1e-8, 0.01, d + i % 3, -1, 0)
            work = torch.empty(lib.ps_tensors_each_workspace_bytes(lists.n), dtype=torch.uint8, device="cuda")
            rc = lib.ps_adam_step_tensors_each(OPT, 1, lists.rows, lists.numels, each, lists.n, scale, state, work.data_ptr(), work.numel(), s)
        else:
            rc = lib.ps_adam_step_tensors(OPT, step, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, lists.rows, lists.numels, lists.n, None, scale, state, s)
        _lib.check(rc, "step")
        if decided == "clean":
            scaler.update_scale(None, operator_calls=lists.n)
    adam_op.destroy_adam(OPT)
    return lists.whole()


@pytest.mark.parametrize("decided", ["host", "clean", "skipped"])
@pytest.mark.parametrize("classes", [0, 3, 60])
@pytest.mark.parametrize("gap", [0, 1, 4])
@pytest.mark.parametrize("shape", SHAPES)
def test_one_launch_leaves_the_bits_of_several(shape, gap, classes, decided):
    sizes = SHAPES[shape]
    arithmetic = _lib.PS_ARITH_TORCH if (gap == 4 and decided != "skipped") else _lib.PS_ARITH_OPERATOR
    scale = 1000.0 if gap == 1 else 2.0**12
    near = _run(sizes, gap, False, decided, classes, arithmetic, scale)
    wide = _run(sizes, gap, True, decided, classes, arithmetic, scale)
    for name, a, b in zip(("p", "m", "v", "h"), near, wide):
        ints = torch.int16 if a.dtype == torch.half else torch.int32
        assert torch.equal(a.view(ints), b.view(ints)), name
