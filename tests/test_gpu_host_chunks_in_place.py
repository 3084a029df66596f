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


def _step(n, offset, fp16_on_host, used, empty_chunks, state, n_slots):
    """One step over two host chunks, with ``empty_chunks`` further ones that hold nothing: what they hold then, and whether
    the staging slots have been written."""
    chunks = [_payloads(n, offset, fp16_on_host, seed) for seed in (1, 2)]
    chunks[1][0][1][used:] = chunks[1][1][1][used:] = chunks[1][2][1][used:] = chunks[1][3][1][used:] = 0.0
    rows = [[view.data_ptr() for _, view in c] for c in chunks]
    rows += [rows[0]] * empty_chunks
    slots = [[torch.full((n,), 7.0, device="cuda:0") for _ in range(3)] + [torch.empty(n, dtype=torch.half, device="cuda:0")] for _ in range(n_slots)]
    used_numel = (ctypes.c_size_t * len(rows))(n, used, *[0] * empty_chunks)
    lib = _lib.load()
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    torch.cuda.synchronize()
    rc = lib.ps_adam_step_hybrid(
        OPT, 1, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, None, 0, _lib.chunk_array(rows), len(rows), n, used_numel,
        _lib.chunk_array([[t.data_ptr() for t in s] for s in slots]), n_slots, _lib.call_pattern(3, 0, 1, max(1, n // 3)) if n > 1 else None,
        1000.0, state, _lib.current_stream_handle(),
    )
    _lib.check(rc, "ps_adam_step_hybrid")
    torch.cuda.synchronize()
    adam_op.destroy_adam(OPT)
    copied = [any(bool((t != 7.0).any()) for t in s[:3]) for s in slots]
    return [[whole.cpu().clone() for whole, _ in c] for c in chunks], copied


@pytest.mark.parametrize("decided", ["host", "device", "skipped"])
@pytest.mark.parametrize("fp16_on_host", [False, True])
@pytest.mark.parametrize("n,offset", [(1, 0), (255, 0), (256, 0), (257, 4), (6267, 0), (4096 + 77, 1), (70001, 2)])
def test_in_place_and_copied_host_chunks_agree_bit_for_bit(n, offset, fp16_on_host, decided):
    got = []
    for empty_chunks, n_slots in ((0, 2), (7, 2), (7, 1)):  # two chunks: in place; nine: through the staging slots, or through one, used again
        state = None
        if decided != "host":
            scaler = DynamicLossScaler(init_scale=1000.0).materialize("cuda:0", betas=(0.9, 0.999))
            if decided == "skipped":
                scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            state = scaler.state_ptr
        chunks, copied = _step(n, offset, fp16_on_host, n - n // 4, empty_chunks, state, n_slots)
        assert copied == [empty_chunks > 0] * n_slots
        got.append(chunks)
    for a, *others in zip(*got):
        for b in others:
            for name, x, y in zip(("fp32 param", "exp_avg", "exp_avg_sq", "fp16"), a, b):
                assert torch.equal(x.view(torch.int16 if x.dtype == torch.half else torch.int32),
                                   y.view(torch.int16 if y.dtype == torch.half else torch.int32)), name


MI = 1 << 20


@pytest.mark.parametrize("n_host,offset,n_resident,in_place", [
    (1, 0, 0, True), (2, 0, 0, True), (8, 0, 0, True), (9, 0, 0, False),
    (2, 0, 8, True), (2, 0, 40, False),  # resident chunks that take as long as the copies would save: 31 of this size
    (1, 1, 0, True), (8, 1, 0, False), (8, 16, 0, False),  # accesses that straddle the link's lines
])
def test_host_chunks_are_updated_in_place_where_that_is_no_slower(n_host, offset, n_resident, in_place):
    """Which route a list takes, told by whether the staging slots have been written, and the same bits on both as for the
    same chunks in HBM."""
    gen = torch.Generator(device="cuda:0").manual_seed(n_host)
    made = [[torch.randn(MI, generator=gen, device="cuda:0") * 0.02, torch.randn(MI, generator=gen, device="cuda:0") * 1e-4,
             (torch.randn(MI, generator=gen, device="cuda:0") * 1e-4).square(), (torch.randn(MI, generator=gen, device="cuda:0") * 4).half()]
            for _ in range(n_host)]
    host = []
    for c in made:
        views = [torch.zeros(MI + 16, pin_memory=True)[offset : offset + MI] for _ in range(3)]
        for v, x in zip(views, c):
            v.copy_(x)
        host.append(views + [c[3].clone()])
    zeros = [torch.zeros(MI, device="cuda:0") for _ in range(3)] + [torch.zeros(MI, dtype=torch.half, device="cuda:0")]
    kept = [[u.clone() for u in zeros] for _ in range(n_resident)]
    resident = [[t.data_ptr() for t in c] for c in kept]
    slots = [[torch.full((MI,), 7.0, device="cuda:0") for _ in range(3)] + [torch.empty(0, dtype=torch.half, device="cuda:0")] for _ in range(2)]
    lib = _lib.load()
    args = (1, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1)
    calls = _lib.call_pattern(n_resident + n_host)
    for opt in (OPT, OPT + 1):
        adam_op.create_adam(opt, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    rows = lambda chunks: _lib.chunk_array([[t.data_ptr() for t in c] for c in chunks])
    rc = lib.ps_adam_step_hybrid(
        OPT, *args, _lib.chunk_array(resident) if resident else None, n_resident, rows(host), n_host, MI, None,
        _lib.chunk_array([[t.data_ptr() for t in s[:3]] + [None] for s in slots]), 2, calls, 1000.0, None, _lib.current_stream_handle(),
    )
    _lib.check(rc, "ps_adam_step_hybrid")
    rc = lib.ps_adam_step_chunks(OPT + 1, *args, rows(made), n_host, MI, None, calls, 1000.0, _lib.current_stream_handle())
    _lib.check(rc, "ps_adam_step_chunks")
    torch.cuda.synchronize()
    for opt in (OPT, OPT + 1):
        adam_op.destroy_adam(opt)
    untouched = all(bool((t == 7.0).all()) for s in slots for t in s[:3])
    assert untouched == in_place
    for got, want in zip(host, made):
        for g, w in zip(got, want):
            as_int = torch.int16 if w.dtype == torch.half else torch.int32
            assert torch.equal(g.cuda().view(as_int), w.view(as_int))
