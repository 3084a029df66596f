"""Memory of momentum and variance exists from when an optimizer asks for it, for the positions it asks for, and once.

The lists are on the meta device: sizes and sharing are the real ones, nothing is allocated."""
import random

import pytest
import torch

import patrickstar_amd as ps
from patrickstar_amd import client as client_module
from patrickstar_amd.client import LIST_CLEARANCE, LIST_PERIOD, LIST_SLACK, list_distance, list_shift

MB = 1 << 20
GAPS = LIST_SLACK + 2 * LIST_CLEARANCE


def held(client):
    """Bytes of the allocations that payloads are views of."""
    storages = {}
    for chunk in client.chunk_list.id_to_chunk_map.values():
        if chunk.payload is not None:
            storage = chunk.payload.untyped_storage()
            storages[storage._cdata] = storage.nbytes()
    return sum(storages.values())


def kept(client):
    """Bytes of the allocations that the client holds on to."""
    return sum({s.untyped_storage()._cdata: s.untyped_storage().nbytes() for s in client._slabs}.values())


@pytest.mark.parametrize("numel", [32 * MB, 24 * MB + 5, 300_001, 300 * MB])
def test_a_client_without_an_optimizer_has_no_memory_for_its_state(numel):
    client = ps.PatrickStarClient(0, numel, device="meta")
    client.append_flat_chunks(2)
    stride = -(-numel // 512) * 512
    assert held(client) == kept(client) == 2 * (2 + 4) * stride


@pytest.mark.parametrize("numel,of_three", [(32 * MB, 3), (24 * MB + 5, 1), (32 * MB, 1), (300_001, 2), (300 * MB, 1)])
def test_state_of_the_positions_an_optimizer_is_given(numel, of_three):
    client = ps.PatrickStarClient(0, numel, device="meta")
    params = client.append_flat_chunks(3)
    before = held(client)
    opt = ps.FP16Adam(client, params[3 - of_three :], loss_scaler=ps.LossScaler(8.0), lr=1e-3)
    stride = -(-numel // 512) * 512
    assert before + 8 * of_three * stride <= held(client) <= before + 8 * of_three * stride + GAPS
    assert kept(client) == held(client)
    m, v = (client.chunk_list[client.positions()[-1].exp_avg].payload, client.chunk_list[client.positions()[-1].exp_avg_sq].payload)
    assert m.numel() == v.numel() == numel and m._base.numel() == v._base.numel() == of_three * stride
    assert opt.state[params[-1]]["exp_avg"] is not None


def test_state_lies_in_the_order_of_the_parameters_chunks():
    client = ps.PatrickStarClient(0, 24 * MB, device="meta")
    params = client.append_flat_chunks(4)
    ps.FP16Adam(client, [params[k] for k in (2, 0, 3, 1)], loss_scaler=ps.LossScaler(8.0), lr=1e-3)
    payload = [[client.chunk_list[cid].payload for cid in (pos.fp32, pos.exp_avg, pos.exp_avg_sq)] for pos in client.positions()]
    for k, (p, m, v) in enumerate(payload):
        assert p.storage_offset() - payload[0][0].storage_offset() == k * 24 * MB
        assert m.storage_offset() - payload[0][1].storage_offset() == v.storage_offset() - payload[0][2].storage_offset() == k * 24 * MB


def test_a_master_chunk_that_is_allocated_again_brings_no_state():
    numel = 32 * MB
    client = ps.PatrickStarClient(0, numel, device="meta")
    params = client.append_flat_chunks(1)
    opt = ps.FP16Adam(client, params, loss_scaler=ps.LossScaler(8.0), lr=1e-3)
    before = held(client)
    client.chunk_list[client.positions()[0].fp32].release_payload()
    client.allocate_payloads()
    assert held(client) == before and opt.state[params[0]]["exp_avg"] is not None


def test_lists_go_without_the_gaps_where_there_is_no_memory_for_them(monkeypatch):
    numel = 32 * MB
    client = ps.PatrickStarClient(0, numel, device="meta")
    params = client.append_flat_chunks(1)
    before = held(client)
    zeros = torch.zeros

    def little_memory(n, **kwargs):
        if n > numel:
            raise torch.OutOfMemoryError("no room")
        return zeros(n, **kwargs)

    monkeypatch.setattr(client_module.torch, "zeros", little_memory)
    ps.FP16Adam(client, params, loss_scaler=ps.LossScaler(8.0), lr=1e-3)
    assert held(client) == before + 8 * numel


def test_the_shift_lays_both_lists_clear_of_the_parameters_within_the_slack():
    rng = random.Random(0)
    for _ in range(4000):
        apart = rng.choice([rng.randrange(-(1 << 38), 1 << 38), rng.randrange(-300, 300) * MB])
        distance = list_distance(rng.randrange(80 * MB, 1 << 30) // 2048 * 2048)
        shift = list_shift(apart, distance)
        assert 0 <= shift <= LIST_SLACK and (apart + shift) % MB == 0
        for at in (apart + shift, apart + shift + distance):
            assert LIST_CLEARANCE <= at % LIST_PERIOD <= LIST_PERIOD - LIST_CLEARANCE
