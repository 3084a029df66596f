"""A C++ exception out of the library, in a call that the binding makes without the interpreter lock, is an error of that
call: raised with the lock held again, and the call is not made a second time by the general path."""
import ctypes
import threading

import pytest
import torch

from patrickstar_amd import _lib, adam_op

pytestmark = pytest.mark.gpu


def test_an_exception_is_an_error_of_the_call(monkeypatch):
    _lib.load()
    from patrickstar_amd import _binding

    throws = ctypes.cast(ctypes.CDLL("libstdc++.so.6")._ZSt17__throw_bad_allocv, ctypes.c_void_p).value  # std::__throw_bad_alloc()
    t = [torch.ones(8, device="cuda") for _ in range(4)]
    args = (7802, 1, 1e-3, 0.9, 0.999, 1e-8, 0.0, True, *t, 8.0)
    with pytest.raises(RuntimeError, match="adam_update: std::bad_alloc"):
        _binding.adam_update(throws, *args)
    raised = []

    def other_thread():
        try:
            _binding.adam_update(throws, *args)
        except RuntimeError as e:
            raised.append(str(e))

    thread = threading.Thread(target=other_thread)
    thread.start()
    thread.join()
    assert raised == ["adam_update: std::bad_alloc"]
    monkeypatch.setattr(_lib.load(), "adam_update", lambda *a: _binding.adam_update(throws, *a))
    monkeypatch.setattr(adam_op, "_update", lambda *a: pytest.fail("made again"))
    with pytest.raises(RuntimeError, match="std::bad_alloc"):
        adam_op.adam_update(*args)
    assert all(bool((x == 1).all()) for x in t)
