"""A device-decided step over some of the tensors with one set of numbers: which calls of the library it makes, seen from the host."""
import ctypes
import os

import pytest
import torch

import patrickstar_amd as ps
from patrickstar_amd import _lib
from test_host_logic import _StepCalls
from test_routes import MI, flat_rows, launches

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="HIP library not built")
CALLS = ["ps_overflow_scan_chunks", "ps_adam_step_tensors", "ps_scaler_update"]


class _Calls(_StepCalls):
    """... but for the questions that the library answers on the host."""

    def ps_tensors_at_once(self, chunks, n_chunks, *others):
        return int(n_chunks <= 64)

    def ps_tensors_each_workspace_bytes(self, n):
        return 64 * n


def _step_over_some(monkeypatch, layers, chunk_numel):
    """(optimizer, library, parameters), one parameter frozen"""
    client = ps.PatrickStarClient(0, chunk_numel, device="cpu")
    model = torch.nn.Sequential(*[torch.nn.Linear(8, 7) for _ in range(layers)])  # 63 elements
    client.register_model(model)
    params = list(model.parameters())
    params[1].requires_grad_(False)
    scaler = ps.DynamicLossScaler()
    optimizer = ps.FP16Adam(client, params, loss_scaler=scaler)
    library = _Calls()
    monkeypatch.setattr(_lib, "current_stream_handle", lambda: None)
    monkeypatch.setattr(_lib, "load", lambda: library)
    monkeypatch.setattr(optimizer, "_lib", library)
    size = ctypes.sizeof(_lib.ps_step_state)
    both = torch.zeros(size + _lib.PS_STEP_SCRATCH_BYTES, dtype=torch.uint8)
    scaler._state, scaler._scratch = both[:size], both[size:]
    return optimizer, library, params


@pytest.mark.parametrize("layers,chunk_numel,calls", [(64, 64, ["ps_adam_step_tensors_dynamic"]), (65, 64, CALLS), (130, 64, CALLS), (130, 1000, ["ps_adam_step_tensors_dynamic"])])
def test_more_chunks_than_one_launch_probes_take_the_three_calls(monkeypatch, layers, chunk_numel, calls):
    """Of 65 chunks on the one call forms constants in a launch of its own: it is a launch longer than the others."""
    optimizer, library, params = _step_over_some(monkeypatch, layers, chunk_numel)

    def made():
        library.names.clear()
        optimizer.step()
        return [name for name in library.names if name in CALLS + ["ps_adam_step_tensors_dynamic"]]

    assert made() == calls and made() == calls
    assert (optimizer._tables[1] > 64) == (calls == CALLS)
    params[1].requires_grad_(True)
    assert made() == []  # whole lists
    params[1].requires_grad_(False)
    assert made() == calls


@pytest.mark.parametrize("sizes,moved,opens", [
    ([256] * 64, False, True), ([256] * 65, False, False), ([1], False, True), ([0, 0], False, False), ([300, 0, 5], False, True), ([300, 7, 5], True, False),
    ([64 * MI] * 4, False, True), ([64 * MI] * 4 + [1], False, False),
])
def test_the_library_says_which_lists_open_with_the_plan(sizes, moved, opens):
    rows = flat_rows(sizes)
    if moved:
        rows[1][2] += 1 << 38
    found = launches("dynamic", rows, sizes, True)  # (which compares the answer with what was launched)
    assert (found[0].name == "open_planned_kernel") == opens


def test_the_addresses_of_the_tensors_are_looked_up_once(monkeypatch):
    """Four views of every tensor: most of the host's part of the first step over some of them."""
    optimizer, library, params = _step_over_some(monkeypatch, 8, 1000)
    looked, rows = [], optimizer._tensor_rows
    monkeypatch.setattr(optimizer, "_tensor_rows", lambda trainable, *slot: looked.append(list(trainable)) or rows(trainable, *slot))
    for k in range(3):
        for p in params:
            optimizer.state[p]["lr"] = 0.5**k
        optimizer.step()
    assert library.names.count("ps_adam_step_tensors_dynamic") == 3 and looked == [params[:1] + params[2:]]
    optimizer.invalidate_tables()
    optimizer.step()
    assert len(looked) == 2 and library.names.count("ps_adam_step_tensors_dynamic") == 4


@pytest.mark.parametrize("arithmetic", ["operator", "torch"])
def test_the_records_of_one_set_of_numbers_are_those_of_every_tensor(monkeypatch, arithmetic):
    optimizer, _, params = _step_over_some(monkeypatch, 8, 1000)
    optimizer.arithmetic = arithmetic
    for p in params:
        for key, value in dict(lr=0.25, betas=[0, 0.5], eps=1, weight_decay=3e-2).items():
            optimizer.state[p][key] = value
    optimizer.step()
    plan = optimizer._tensors_of(optimizer._plan)
    general = {key: value for key, value in plan.items() if key != "rows"}
    a, b = [optimizer._each_table(dict(one, table=None)) for one in (plan, general)]
    assert bytes(a[3]) == bytes(b[3]) and len(bytes(a[3])) == 56 * 15
    assert a[:3] == b[:3] and a[4:] == b[4:] and a[5] == (15 if arithmetic == "operator" else 0)
