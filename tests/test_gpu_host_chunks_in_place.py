"""Host-resident chunks that the step's kernel updates where they are (few of them), against the same chunks copied
through staging slots (many of them): same bits, wherever in their allocations the payloads start, whole and part-filled,
for host-decided, device-decided and skipped steps."""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
OPT = 7301


def _payloads(n, offset, fp16_on_host, seed):
    """fp32 param, exp_avg, exp_avg_sq (pinned) and fp16 gradient of one chunk, each ``offset`` elements into its allocation."""
    gen = torch.Generator().manual_seed(seed)
    made = [torch.randn(n, generator=gen) * 0.02, torch.randn(n, generator=gen) * 1e-4,
            (torch.randn(n, generator=gen) * 1e-4).square(), (torch.randn(n, generator=gen) * 4).half()]
    out = []
    for k, x in enumerate(made):
        on_host = k < 3 or fp16_on_host
        whole = torch.zeros(n + 8, dtype=x.dtype, pin_memory=True) if on_host else torch.zeros(n + 8, dtype=x.dtype, device="cuda:0")
        whole[offset : offset + n] = x
        out.append((whole, whole[offset : offset + n]))
    return out


def _step(n, offset, fp16_on_host, used, empty_chunks, state):
    """One step over two host chunks, with ``empty_chunks`` further ones that hold nothing."""
    chunks = [_payloads(n, offset, fp16_on_host, seed) for seed in (1, 2)]
    chunks[1][0][1][used:] = chunks[1][1][1][used:] = chunks[1][2][1][used:] = chunks[1][3][1][used:] = 0.0
    rows = [[view.data_ptr() for _, view in c] for c in chunks]
    rows += [rows[0]] * empty_chunks
    slots = [[torch.empty(n, device="cuda:0") for _ in range(3)] + [torch.empty(n, dtype=torch.half, device="cuda:0")] for _ in range(2)]
    used_numel = (ctypes.c_size_t * len(rows))(n, used, *[0] * empty_chunks)
    lib = _lib.load()
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    torch.cuda.synchronize()
    rc = lib.ps_adam_step_hybrid(
        OPT, 1, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, None, 0, _lib.chunk_array(rows), len(rows), n, used_numel,
        _lib.chunk_array([[t.data_ptr() for t in s] for s in slots]), 2, _lib.call_pattern(3, 0, 1, max(1, n // 3)) if n > 1 else None,
        1000.0, state, _lib.current_stream_handle(),
    )
    _lib.check(rc, "ps_adam_step_hybrid")
    torch.cuda.synchronize()
    adam_op.destroy_adam(OPT)
    return [[whole.cpu().clone() for whole, _ in c] for c in chunks]


@pytest.mark.parametrize("decided", ["host", "device", "skipped"])
@pytest.mark.parametrize("fp16_on_host", [False, True])
@pytest.mark.parametrize("n,offset", [(1, 0), (255, 0), (256, 0), (257, 4), (6267, 0), (4096 + 77, 1), (70001, 2)])
def test_in_place_and_copied_host_chunks_agree_bit_for_bit(n, offset, fp16_on_host, decided):
    got = []
    for empty_chunks in (0, 7):  # two chunks: in place; nine: through the staging slots
        state = None
        if decided != "host":
            scaler = DynamicLossScaler(init_scale=1000.0).materialize("cuda:0", betas=(0.9, 0.999))
            if decided == "skipped":
                scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            state = scaler.state_ptr
        got.append(_step(n, offset, fp16_on_host, n - n // 4, empty_chunks, state))
    for a, b in zip(*got):
        for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a, b):
            assert torch.equal(x.view(torch.int16 if x.dtype == torch.half else torch.int32),
                               y.view(torch.int16 if y.dtype == torch.half else torch.int32)), name
