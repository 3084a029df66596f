"""Chunks at one distance from one another take kernels whose addresses are preloaded; any other list takes the general ones.  The
same chunks listed in the opposite order are such another list, and have to be left with the same bits: lengths around the ends
of tiles, a shorter last chunk, more chunks than one general launch takes, spans of the first call that cut tiles, every
decision and both arithmetics."""
import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
T = 256
OPT = 8001

# chunks, elements of a chunk, elements of the last one, span of the first call (chunk, offset, elements; None: one call)
LISTS = {
    "two": (2, 5 * T, 5 * T, None),
    "short_list": (3, 25 * T + 3, 20 * T - 1, (1, 2 * T + 1, 5 * T)),
    "short_list_of_64": (64, T, 5, (63, 1, 3)),
    "ragged": (3, 33 * T + 77, 33 * T + 77, (1, 100, 3 * T)),
    "short_last": (4, 100 * T + 1, 100 * T - 255, (3, 0, 7)),
    "empty_last": (3, 90 * T, 0, (0, 0, 90 * T)),
    "one_left": (2, 81 * T, 1, (1, 0, 1)),
    "many": (70, 2 * T + 9, T, (69, 13, 200)),
    "span_at_tiles": (2, 300 * T, 299 * T, (0, T, 4 * T)),
}


def _run(name, mirrored, decided, arithmetic, scale, eps, adamw, wd):
    lib, s = _lib.load(), _lib.current_stream_handle()
    chunks, n, last, span = LISTS[name]
    stride = -(-n // 512) * 512
    gen = torch.Generator(device="cuda").manual_seed(chunks)
    data = [torch.randn(chunks * stride, device="cuda", generator=gen) * f for f in (0.02, 1e-4, 1e-3)]
    data[2].square_()
    data.append((torch.randn(chunks * stride, device="cuda", generator=gen) * 1e-3 * scale).half())
    for t in data:
        t.view(chunks, stride)[:, n:] = 0
        t.view(chunks, stride)[-1, last:] = 0
    if decided.endswith("flagged"):
        data[3].view(chunks, stride)[0, n // 2] = float("inf")
    order = list(range(chunks))[:: -1 if mirrored else 1]
    rows = _lib.chunk_array([[t.view(chunks, stride)[k].data_ptr() for t in data] for k in order])
    used = _lib.size_array([last if k == chunks - 1 else n for k in order])
    calls = None
    if span is not None and arithmetic == _lib.PS_ARITH_OPERATOR:
        calls = _lib.call_pattern(5, order.index(span[0]), span[1], span[2])
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, eps, wd, adamw, False)
    lib.ps_adam_set_arithmetic(OPT, arithmetic)
    lib.ps_adam_set_grad_clamp(OPT, 0.5)
    scaler = None
    if decided != "host":
        scaler = DynamicLossScaler(init_scale=scale).materialize("cuda:0", betas=(0.9, 0.999))
    for step in (1, 2):
        if scaler is None:
            rc = lib.ps_adam_step_chunks(OPT, step, 1e-3, 0.9, 0.999, eps, wd, 1, rows, chunks, n, used, calls, scale, s)
        elif decided.startswith("dynamic"):
            rc = lib.ps_adam_step_chunks_dynamic(OPT, 1e-3, eps, wd, 1, rows, chunks, n, used, calls, 1, scaler.state_ptr, None, 0,
                                                 5 if calls is not None else 1, s)
        else:
            _lib.check(lib.ps_overflow_scan_chunks(rows, chunks, n, used, scaler.state_ptr, s), "scan")
            rc = lib.ps_adam_step_chunks_gated(OPT, 1e-3, eps, wd, 1, rows, chunks, n, used, calls, scaler.state_ptr, s)
        _lib.check(rc, "step")
        if scaler is not None and not decided.startswith("dynamic"):
            assert scaler.overflow_flag == (decided == "flagged" and step == 1)
            scaler.update_scale(None, operator_calls=5 if calls is not None else 1)
    adam_op.destroy_adam(OPT)
    if scaler is not None:
        data.append(scaler._state.clone())
    return data


@pytest.mark.parametrize("decided", ["host", "clean", "flagged", "dynamic", "dynamic flagged"])
@pytest.mark.parametrize(
    "arithmetic,scale,eps,adamw,wd",
    [(0, 2.0**12, 1e-8, True, 0.01), (0, 1000.0, 1e-8, False, 0.01), (0, 2.0**8, 0.0, True, 0.0), (1, 1000.0, 1e-8, True, 0.01)],
)
@pytest.mark.parametrize("name", LISTS)
def test_preloaded_addresses_leave_the_bits_of_descriptors(name, arithmetic, scale, eps, adamw, wd, decided):
    even = _run(name, False, decided, arithmetic, scale, eps, adamw, wd)
    general = _run(name, True, decided, arithmetic, scale, eps, adamw, wd)
    for what, a, b in zip(("p", "m", "v", "h", "state"), even, general):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what
