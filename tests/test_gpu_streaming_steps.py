"""Long lists whose tiles fill whole 64-byte lines are stepped and probed with the non-temporal hint, by kernels of their own; the
same numbers at a phase of 32 bytes take the others and have to be left with the same bits.  (That these lists take two routes is
checked in test_routes.py.)"""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
MI = 1 << 20
OPT = 8101


def _lists(n, phase, scale, poison=None):
    gen = torch.Generator(device="cuda").manual_seed(n % 1000)
    out = []
    for k, f in enumerate((0.02, 1e-4, 1e-3, 1e-3 * scale)):
        whole = torch.empty(n + 64, device="cuda").normal_(0, f, generator=gen)
        whole = whole.square_() if k == 2 else whole.half() if k == 3 else whole
        out.append(torch.empty_like(whole)[phase : phase + n].copy_(whole[:n]))
    if poison is not None:
        out[3][poison] = float("inf")
    return out


def _same(a, b):
    for what, x, y in zip(("p", "m", "v", "h", "state"), a, b):
        ints = {torch.half: torch.int16, torch.float: torch.int32}.get(x.dtype)
        assert torch.equal(x if ints is None else x.view(ints), y if ints is None else y.view(ints)), what


def _scaler(decided, scale):
    return None if decided == "host" else DynamicLossScaler(init_scale=scale).materialize("cuda:0", betas=(0.9, 0.999))


@pytest.mark.parametrize("arithmetic,scale,adamw,wd", [(0, 2.0**12, True, 0.01), (0, 1000.0, False, 0.01), (1, 1000.0, False, 0.0)])
@pytest.mark.parametrize("decided", ["host", "device", "flagged"])
@pytest.mark.parametrize("numel,chunks,mirrored", [(33 * MI + 77, 1, False), (17 * MI, 2, False), (17 * MI, 2, True)])
def test_chunk_lists(numel, chunks, mirrored, decided, arithmetic, scale, adamw, wd):
    lib, s, got = _lib.load(), _lib.current_stream_handle(), []
    for phase in (0, 16):  # 16: 64 bytes of fp32, 32 of fp16
        lists = _lists(numel * chunks, phase, scale, numel * chunks - 1 if decided == "flagged" else None)
        order = range(chunks)[:: -1 if mirrored else 1]
        rows = _lib.chunk_array([[t[k * numel :].data_ptr() for t in lists] for k in order])
        calls = None if arithmetic else _lib.call_pattern(7, 0, 1000, 5 * MI + 3)
        adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, wd, adamw, False)
        lib.ps_adam_set_arithmetic(OPT, arithmetic)
        scaler = _scaler(decided, scale)
        for step in (1, 2):
            if scaler is None:
                rc = lib.ps_adam_step_chunks(OPT, step, 1e-3, 0.9, 0.999, 1e-8, wd, 1, rows, chunks, numel, None, calls, scale, s)
            else:
                rc = lib.ps_adam_step_chunks_dynamic(OPT, 1e-3, 1e-8, wd, 1, rows, chunks, numel, None, calls, 1, scaler.state_ptr, None, 0, 7, s)
            _lib.check(rc, "step")
        adam_op.destroy_adam(OPT)
        if scaler is not None:
            state = _lib.ps_step_state()
            _lib.check(lib.ps_state_read(scaler.state_ptr, ctypes.byref(state), s), "ps_state_read")
            assert state.skipped_steps == (1 if decided == "flagged" else 0)
            lists.append(scaler._state.clone())
        got.append(lists)
    _same(*got)


@pytest.mark.parametrize("each", [False, True])
@pytest.mark.parametrize("decided", ["host", "device", "flagged"])
@pytest.mark.parametrize("moved", [False, True])  # one tensor's variance elsewhere: several launches by length
def test_tensor_lists(moved, decided, each):
    sizes = [20 * MI, 3, 6 * MI + 1, 255, 6 * MI - 7, 1 * MI, 256, 500_000]
    lib, s, got, n, scale = _lib.load(), _lib.current_stream_handle(), [], sum(sizes), 2.0**12
    for phase in (0, 8):  # of momentum and variance alone
        lists = _lists(n, 0, scale)
        lists[1], lists[2] = (torch.empty(n + 64, device="cuda")[phase : phase + n].copy_(t) for t in lists[1:3])
        at = [sum(sizes[:i]) for i in range(len(sizes))]
        rows = [[t[a:].data_ptr() for t in lists] for a in at]
        own = torch.empty(sizes[-1] + 256, device="cuda")
        if moved:
            k = (lists[2][at[-1] :].data_ptr() - own.data_ptr()) // 4 % 256  # at the same phase of a KiB
            own = own[k : k + sizes[-1]].copy_(lists[2][at[-1] :])
            rows[-1][2] = own.data_ptr()
        numels = (ctypes.c_size_t * len(sizes))(*sizes)
        adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
        scaler = _scaler(decided, scale)
        if decided == "flagged":
            scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
        state = scaler.state_ptr if scaler is not None else None
        if each:
            calls = (_lib.ps_tensor_call * len(sizes))(*[(1e-3 * (i + 1), 0.9, 0.999, 1e-8, 0.01, 4 if scaler is None else i % 2, -1, 0) for i in range(len(sizes))])
            work = torch.empty(lib.ps_tensors_each_workspace_bytes(len(sizes)), dtype=torch.uint8, device="cuda")
            rc = lib.ps_adam_step_tensors_each(OPT, 1, _lib.chunk_array(rows), numels, calls, len(sizes), scale, state, work.data_ptr(), work.numel(), s)
        else:
            rc = lib.ps_adam_step_tensors(OPT, 4, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, _lib.chunk_array(rows), numels, len(sizes), None, scale, state, s)
        _lib.check(rc, "step")
        adam_op.destroy_adam(OPT)
        if moved:
            lists[2][at[-1] :] = own
        got.append(lists)
    _same(*got)


@pytest.mark.parametrize("half,out", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("n,head", [(256 * 1024, 0), (256 * 1024 - 1, 0), (300_001, 3), (2 * MI + 255, 128)])
def test_operator(n, head, half, out):
    lib, s, got = _lib.load(), _lib.current_stream_handle(), []
    for phase in (0, 8):  # of momentum and variance alone
        lists = _lists(n + 256, 0, 8.0)
        at = (256 - head) % 256
        m, v = (torch.empty(n + 512, device="cuda")[phase : phase + n + 256].copy_(t) for t in lists[1:3])
        g = lists[3] if half else lists[3].float()
        h = torch.zeros(n + 256, dtype=torch.half, device="cuda")
        adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
        rc = lib.ps_adam_update(OPT, 3, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, lists[0][at:].data_ptr(), g[at:].data_ptr(), int(half),
                                m[at:].data_ptr(), v[at:].data_ptr(), n, 8.0, h[at:].data_ptr() if out else None, s)
        _lib.check(rc, "ps_adam_update")
        adam_op.destroy_adam(OPT)
        got.append([lists[0], m, v, h])
    _same(*got)
