"""The restore of a skipped step, which a quarter of the update's workgroups do: lengths around the ends of the groups they
lead, chunks of different lengths in one launch, tensors with elements in front of their tile grid.  Every fp16 element
becomes its master rounded to nearest even, nothing else changes."""
import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
OPT = 7601
T = 256  # elements per tile; leaders: 32 of 128 workgroups, 4 tiles each

LENGTHS = [1, T, 31 * T + 5, 32 * T, 33 * T, 96 * T, 97 * T + 1, 127 * T, 128 * T, 128 * T + 1, 129 * T + 7, 160 * T, 512 * T + 77, 1000 * T - 1]


def _flagged():
    scaler = DynamicLossScaler(init_scale=2.0**8).materialize("cuda:0", betas=(0.9, 0.999))
    scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
    return scaler


def _lists(total, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lists = [torch.randn(total, device="cuda", generator=gen) for _ in range(3)]
    return lists + [torch.full((total,), 7.0, dtype=torch.half, device="cuda")]


def _check(lists, before, spans):
    for a, b in zip(lists[:3], before[:3]):
        assert torch.equal(a, b)
    want = before[3]
    for lo, hi in spans:
        want[lo:hi] = before[0][lo:hi].half()
    assert torch.equal(lists[3].view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("offset", [0, 1, 4])
@pytest.mark.parametrize("used", [[n] for n in LENGTHS] + [LENGTHS, LENGTHS[::-1], [0, 129 * T + 7, 0, 5]], ids=str)
def test_chunk_lists(used, offset):
    n = max(used)
    stride = n + 64 - n % 8
    lists = _lists(len(used) * stride + 8, len(used))
    before = [t.clone() for t in lists]
    rows = [[t[i * stride + offset :].data_ptr() for t in lists] for i in range(len(used))]
    scaler = _flagged()
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    rc = _lib.load().ps_adam_step_chunks_gated(OPT, 1e-3, 1e-8, 0.01, 1, _lib.chunk_array(rows), len(used), n, _lib.size_array(used),
                                               None, scaler.state_ptr, _lib.current_stream_handle())
    _lib.check(rc, "gated")
    adam_op.destroy_adam(OPT)
    _check(lists, before, [(i * stride + offset, i * stride + offset + u) for i, u in enumerate(used)])


@pytest.mark.parametrize("each", [False, True])
@pytest.mark.parametrize("gap", [0, 1, 7, 100])  # 0: one tensor right behind the other, at every phase of a KiB
def test_tensor_lists(gap, each):
    lists = _lists(sum(LENGTHS) + (gap + 8) * len(LENGTHS) + 300, gap)
    before = [t.clone() for t in lists]
    spans, at = [], 3
    for n in LENGTHS:
        spans.append((at, at + n))
        at += n + gap
    rows = _lib.chunk_array([[t[lo:].data_ptr() for t in lists] for lo, _ in spans])
    numels, count = _lib.size_array(LENGTHS), len(LENGTHS)
    scaler, lib, s = _flagged(), _lib.load(), _lib.current_stream_handle()
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    if each:
        calls = (_lib.ps_tensor_call * count)(*[(1e-3, 0.9, 0.999, 1e-8, 0.01, i % 2, 0, 0) for i in range(count)])
        work = torch.empty(lib.ps_tensors_each_workspace_bytes(count), dtype=torch.uint8, device="cuda")
        rc = lib.ps_adam_step_tensors_each(OPT, 1, rows, numels, calls, count, -1.0, scaler.state_ptr, work.data_ptr(), work.numel(), s)
    else:
        rc = lib.ps_adam_step_tensors(OPT, 0, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, rows, numels, count, None, -1.0, scaler.state_ptr, s)
    _lib.check(rc, "tensors")
    adam_op.destroy_adam(OPT)
    _check(lists, before, spans)
