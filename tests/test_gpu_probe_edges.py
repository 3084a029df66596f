"""The inf/nan probe at the edges of its tiles: lengths around whole vectors and whole tiles, buffers that start off a
16-byte boundary, and non-finite neighbours just outside the buffer, which it must not see."""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, _lib

pytestmark = pytest.mark.gpu

# vectors of 8 halves / 4 floats, tiles of 4096 halves / 2048 floats, 8192 halves in the allocation-free form
LENGTHS = [1, 3, 7, 8, 9, 63, 512, 2047, 2048, 2049, 4095, 4096, 4097, 6267, 8191, 8192, 8193, 20001]


def _flag(scaler):
    return scaler.overflow_flag


@pytest.mark.parametrize("offset", [0, 1, 2, 5])
@pytest.mark.parametrize("dtype", [torch.half, torch.float])
def test_probe_sees_every_element_of_the_buffer_and_none_outside(dtype, offset):
    scaler = DynamicLossScaler(init_scale=1).materialize("cuda:0")
    word = torch.zeros(1, dtype=torch.int32, device="cuda:0")
    for n in LENGTHS:
        whole = torch.full((n + 64,), float("inf"), dtype=dtype, device="cuda:0")
        x = whole[16 + offset : 16 + offset + n]
        x.fill_(65504.0)

        def clean():
            scaler._state[_lib.ps_step_state.overflow.offset :][:4].zero_()
            word.zero_()

        def probe():
            """(flag of the tensor form, flag of the allocation-free chunk form)"""
            clean()
            scaler.scan(x)
            if dtype == torch.half:
                row = _lib.chunk_array([[16, 16, 16, x.data_ptr()]])
                rc = _lib.load().ps_overflow_scan_chunks_noalloc(row, 1, n, word.data_ptr(), _lib.current_stream_handle())
                _lib.check(rc, "ps_overflow_scan_chunks_noalloc")
                one = _flag(scaler)
                clean_state = bool(word.item())
                # the chunk-list form, over the used part of a longer chunk
                scaler._state[_lib.ps_step_state.overflow.offset :][:4].zero_()
                used = (ctypes.c_size_t * 1)(n)
                rc = _lib.load().ps_overflow_scan_chunks(row, 1, n + 32, used, scaler.state_ptr, _lib.current_stream_handle())
                _lib.check(rc, "ps_overflow_scan_chunks")
                return one, clean_state, _flag(scaler)
            return (_flag(scaler),)

        assert not any(probe()), f"n = {n}: saw a neighbour"
        for at in sorted({0, n - 1, n // 2, max(0, n - 9), min(n - 1, 8)}):
            keep = x[at].clone()
            for bad in (float("inf"), float("-inf"), float("nan")):
                x[at] = bad
                assert all(probe()), f"n = {n}: missed {bad} at {at}"
            x[at] = keep
