"""Tensors with binary32 gradients among a list that streams past the caches, and a large one beside a list that does not: the same
bits as the two kinds stepped in calls of their own (which of them takes the hint is checked in test_routes.py)."""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
MI = 1 << 20
OPT = 8201


def _tensors(sizes, scale, phases):
    gen = torch.Generator(device="cuda").manual_seed(sum(n for n, _ in sizes) % 1000)
    out = []
    for (n, wide), phase in zip(sizes, phases):
        p, m, v, g = (torch.empty(n + 64, device="cuda").normal_(0, f, generator=gen)[phase : phase + n] for f in (0.02, 1e-4, 1e-3, 1e-3 * scale))
        out.append([p, m, v.square_(), g if wide else torch.empty(n + 64, dtype=torch.half, device="cuda")[phase : phase + n].copy_(g)])
    return out


def _step(tensors, wide, scaler, scale):
    lib, s, n = _lib.load(), _lib.current_stream_handle(), len(tensors)
    each = (_lib.ps_tensor_call * n)(*[(1e-3, 0.9, 0.999, 1e-8, 0.01, 4 if scaler is None else 0, -1, int(w)) for w in wide])
    work = torch.empty(lib.ps_tensors_each_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    rows = _lib.chunk_array([[t.data_ptr() for t in ts] for ts in tensors])
    rc = lib.ps_adam_step_tensors_each(OPT, 1, rows, (ctypes.c_size_t * n)(*[ts[0].numel() for ts in tensors]), each, n, scale,
                                       scaler.state_ptr if scaler is not None else None, work.data_ptr(), work.numel(), s)
    _lib.check(rc, "step")
    adam_op.destroy_adam(OPT)


@pytest.mark.parametrize("decided", ["host", "device"])
@pytest.mark.parametrize(
    "sizes,phases",
    [([(33 * MI, False), (300_001, True), (2 * MI + 1, False)], (0, 4, 16)),  # long, and a binary32 gradient off the lines
     ([(MI, False), (40 * MI, True), (255, True), (70_001, False)], (0, 0, 1, 0))],  # short, and a large one
)
def test_the_same_bits_as_in_calls_of_their_own(sizes, phases, decided):
    scale, wide = 2.0**12, [w for _, w in sizes]
    got = []
    for apart in (False, True):
        tensors = _tensors(sizes, scale, phases)
        scaler = None if decided == "host" else DynamicLossScaler(init_scale=scale).materialize("cuda:0", betas=(0.9, 0.999))
        if not apart:
            _step(tensors, wide, scaler, scale)
        else:
            for kind in (False, True):
                of_kind = [ts for ts, w in zip(tensors, wide) if w == kind]
                other = None if scaler is None else DynamicLossScaler(init_scale=scale).materialize("cuda:0", betas=(0.9, 0.999))
                _step(of_kind, [kind] * len(of_kind), other, scale)
        got.append([t for ts in tensors for t in ts])
    for x, y in zip(*got):
        ints = torch.int16 if x.dtype == torch.half else torch.int32
        assert torch.equal(x.contiguous().view(ints), y.contiguous().view(ints))
