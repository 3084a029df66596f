"""The probe of a long list reads its beginning through the caches and the rest past them: an inf or a nan on either side of the lines, and at
the ends of the list, is found; none is found where there is none."""
import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib, adam_op

pytestmark = pytest.mark.gpu
MI = 1 << 20
KEEP, LONG, KEEP_LONG = 112 * MI, 256 * MI, 64 * MI
OPT = 8501


def _flag(scaler):
    return scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32)


# chunks, elements of each, elements of the last, distance in front of the second one beyond its place
@pytest.mark.parametrize("chunks,n,last,apart", [(1, KEEP, KEEP, 0), (1, KEEP + 1, KEEP + 1, 0), (3, 40 * MI + 8, 35 * MI + 3, 0), (3, 40 * MI + 8, 35 * MI + 3, 8),
                                                 (70, 2 * MI + 5, 77, 0), (2, LONG // 2, LONG // 2, 0), (2, LONG // 2 + 8, LONG // 2 + 1, 0)])
def test_scan(chunks, n, last, apart):
    lib, s = _lib.load(), _lib.current_stream_handle()
    h = torch.zeros(chunks * n + apart, dtype=torch.half, device="cuda")
    at = [k * n + (apart if k else 0) for k in range(chunks)]
    other = h.data_ptr()  # the probe looks at the fp16 lists only
    table = _lib.chunk_array([(other, other, other, h[a:].data_ptr()) for a in at])
    used = _lib.size_array([n] * (chunks - 1) + [last])
    scaler = DynamicLossScaler(init_scale=8.0).materialize("cuda:0", betas=(0.9, 0.999))
    end = at[-1] + last - 1
    places = [p for p in (0, KEEP - 1, KEEP, KEEP_LONG - 1, KEEP_LONG, KEEP_LONG + 1, n - 1, end // 2, end) if p <= end and any(a <= p < a + n for a in at)]
    for place in [None, *places, None]:
        if place is not None:
            h[place] = float("nan") if place % 2 else float("inf")
        _lib.check(lib.ps_overflow_scan_chunks(table, chunks, n, used, scaler.state_ptr, s), "scan")
        assert int(_flag(scaler)) == (place is not None), place
        _flag(scaler).zero_()
        if place is not None:
            h[place] = 0


@pytest.mark.parametrize("each", [False, True])
def test_whole_steps(each):
    lib, s, n = _lib.load(), _lib.current_stream_handle(), KEEP + 4099
    lists = [torch.full((n,), f, device="cuda", dtype=t) for f, t in ((0.5, torch.float), (1e-3, torch.float), (1e-4, torch.float), (0.25, torch.half))]
    table = _lib.chunk_array([[t.data_ptr() for t in lists]])
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    scaler = DynamicLossScaler(init_scale=8.0).materialize("cuda:0", betas=(0.9, 0.999))
    calls = (_lib.ps_tensor_call * 1)(_lib.ps_tensor_call(1e-3, 0.9, 0.999, 1e-8, 0.01, 0, -1, 0))
    work = torch.empty(lib.ps_tensors_each_workspace_bytes(1), dtype=torch.uint8, device="cuda")
    scratch = (scaler._scratch.data_ptr(), _lib.PS_STEP_SCRATCH_BYTES)
    skipped = 0
    for place in (None, KEEP - 1, KEEP, n - 1, None):
        lists[3].fill_(0.25)
        if place is not None:
            lists[3][place] = float("inf")
            skipped += 1
        if each:
            rc = lib.ps_adam_step_tensors_dynamic(OPT, 1, table, 1, n, None, table, _lib.size_array([n]), calls, 1, scaler.state_ptr, None, 0, 1,
                                                  work.data_ptr(), work.numel(), *scratch, s)
        else:
            rc = lib.ps_adam_step_chunks_dynamic_scratch(OPT, 1e-3, 1e-8, 0.01, 1, table, 1, n, None, None, 1, scaler.state_ptr, None, 0, 1, *scratch, s)
        _lib.check(rc, "step")
        assert scaler.skipped_steps == skipped, place
        for t in lists[:3]:
            assert bool((t == t[0]).all())
    adam_op.destroy_adam(OPT)
