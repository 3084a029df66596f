"""The device-decided step in one call: a short chunk list (one launch) and lists on both sides of the line, against the
probe, the step and the scale update as calls of their own: payloads, step state and log the same bits."""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
OPT = 7501
TILES = 80  # of 256 elements: the longest list that is one launch

# chunks, chunk length, used lengths (None: all full), element offset of the payloads in their allocations
LISTS = [
    (1, 1, None, 0), (1, 256, None, 0), (3, 6267, None, 0), (1, TILES * 256, None, 0), (1, TILES * 256 + 1, None, 0),
    (7, 4111, [4111, 4000, 256, 255, 1, 0, 4111], 0), (64, 300, None, 4), (65, 255, None, 0), (2, 5000, [4097, 300], 1),
    (8, 10 * 256, None, 0), (8, 10 * 256 + 1, None, 0),
]


class _Run:
    def __init__(self, one_call, case, arithmetic, adamw, wd, clamp, scale, eps):
        self.one_call, self.case, self.eps, self.wd = one_call, case, eps, wd
        n_chunks, n, used, offset = case
        gen = torch.Generator(device="cuda").manual_seed(n_chunks * n)
        self.lists = []
        for std, dt in ((0.02, torch.float), (1e-4, torch.float), (1e-4, torch.float), (3.0, torch.half)):
            whole = torch.zeros(n_chunks, n + 8 + offset, device="cuda", dtype=dt)
            for i in range(n_chunks):
                u = n if used is None else used[i]
                whole[i, offset : offset + u] = (torch.randn(u, device="cuda", generator=gen) * std).to(dt)
            self.lists.append(whole)
        self.lists[2].square_()
        self.table = _lib.chunk_array([[t[i, offset:].data_ptr() for t in self.lists] for i in range(n_chunks)])
        self.used = _lib.size_array(used)
        self.scaler = DynamicLossScaler(init_scale=scale, scale_window=2, min_scale=1).materialize("cuda:0", betas=(0.9, 0.999))
        self.scaler.enable_log(4)
        adam_op.create_adam(OPT + one_call, 1e-3, 0.9, 0.999, eps, wd, adamw, False)
        lib = _lib.load()
        if clamp:
            _lib.check(lib.ps_adam_set_grad_clamp(OPT + one_call, clamp), "clamp")
        _lib.check(lib.ps_adam_set_arithmetic(OPT + one_call, arithmetic), "arithmetic")

    def step(self, probe, operator_calls, span):
        n_chunks, n, used, _ = self.case
        lib, s = _lib.load(), _lib.current_stream_handle()
        calls = _lib.call_pattern(operator_calls, *span) if operator_calls else None
        args = (1e-3, self.eps, self.wd, 1, self.table, n_chunks, n, self.used, calls)
        state = self.scaler.state_ptr
        if self.one_call:
            _lib.check(lib.ps_adam_step_chunks_dynamic(OPT + 1, *args, int(probe), state, *self.scaler.log_arguments(), operator_calls, s), "one call")
            return
        if probe:
            _lib.check(lib.ps_overflow_scan_chunks(self.table, n_chunks, n, self.used, state, s), "scan")
        _lib.check(lib.ps_adam_step_chunks_gated(OPT, *args, state, s), "gated")
        self.scaler.update_scale(None, operator_calls=operator_calls)


@pytest.mark.parametrize("case", LISTS, ids=[f"{c[0]}x{c[1]}" for c in LISTS])
@pytest.mark.parametrize("arithmetic,adamw,wd,clamp,scale,eps", [
    (0, True, 0.01, 0.0, 2.0**12, 1e-8), (0, False, 0.01, 1.0, 1000.0, 1e-8), (1, True, 0.0, 0.0, 2**16, 1e-8), (0, True, 0.01, 0.0, 2.0**12, 0.0),
])
def test_one_call_is_its_three_parts(case, arithmetic, adamw, wd, clamp, scale, eps):
    runs = [_Run(one, case, arithmetic, adamw, wd, clamp, scale, eps) for one in (False, True)]
    n_chunks, n, used, offset = case
    last = max(i for i in range(n_chunks) if used is None or used[i])
    span = (last, 0, (n if used is None else used[last]) // 2)
    # a clean step, an overflow that only the probe can see, one that only the flag knows of, clean steps again
    for k, (poison, probe, flag) in enumerate([(0, 1, 0), (1, 1, 0), (0, 0, 1), (0, 0, 0), (0, 1, 0)]):
        for r in runs:
            u = n if used is None else used[last]
            grads = r.lists[3]
            grads[:, offset : offset + n] = torch.where(r.lists[0][:, offset : offset + n] == 0, 0.0, grads[:, offset : offset + n] * 50).half()
            if poison:
                grads[last, offset + u - 1] = float("nan") if k % 2 else float("inf")
            if flag:
                r.scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            r.step(probe, 0 if arithmetic else (1 if k == 3 else 3), (0, 0, 0) if k == 3 else span)
        a, b = runs
        for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a.lists, b.lists):
            kind = torch.int16 if x.dtype == torch.half else torch.int32
            assert torch.equal(x.view(kind), y.view(kind)), (k, name)
        assert torch.equal(a.scaler._state, b.scaler._state), k
        assert torch.equal(a.scaler._log, b.scaler._log), k
    for one in (0, 1):
        adam_op.destroy_adam(OPT + one)


def test_one_call_refuses_what_its_parts_refuse():
    lib = _lib.load()
    r = _Run(1, (1, 300, None, 0), 0, True, 0.01, 0.0, 2.0**12, 1e-8)
    state, s = r.scaler.state_ptr, _lib.current_stream_handle()
    before = [t.clone() for t in r.lists] + [r.scaler._state.clone()]
    used, E = (ctypes.c_size_t * 1)(301), _lib.PS_ERR_BAD_ARG
    f = lib.ps_adam_step_chunks_dynamic
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, None, None, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, None, 1, 300, None, None, 1, state, None, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, -1, 300, None, None, 1, state, None, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, used, None, 1, state, None, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, _lib.call_pattern(3, 1, 0, 1), 1, state, None, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, state, 0, 1, s) == E
    assert f(OPT + 1, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, None, 0, -1, s) == E
    assert f(4711, 1e-3, 1e-8, 0.0, 1, r.table, 1, 300, None, None, 1, state, None, 0, 1, s) == _lib.PS_ERR_UNKNOWN_ID
    torch.cuda.synchronize()
    for a, b in zip(before, r.lists + [r.scaler._state]):
        assert torch.equal(a, b)
    adam_op.destroy_adam(OPT + 1)
