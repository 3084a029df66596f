"""Where the fp32 lists start against one another: the distance rule, and that every chunk has its own zero-filled memory."""
import pytest
import torch

import patrickstar_amd as ps
from patrickstar_amd.chunk_layout import AccessType, ChunkType, ParamType, register_param
from patrickstar_amd.client import LIST_CLEARANCE, LIST_PERIOD, list_distance

MB = 1 << 20


@pytest.mark.parametrize(
    "nbytes", [80 * MB, 128 * MB - 4, 128 * MB, 128 * MB + 2048, 137 * MB - 2048, 137 * MB, 183 * MB, 183 * MB + 2048, 192 * MB - 2048, 1 << 30]
)
def test_neither_the_distance_nor_its_double_is_nearly_a_multiple_of_128_MiB(nbytes):
    d = list_distance(nbytes)
    assert nbytes <= d <= nbytes + 2 * LIST_CLEARANCE
    for distance in (d, 2 * d):
        past = distance % (128 * MB)
        assert LIST_CLEARANCE <= past <= 128 * MB - LIST_CLEARANCE
    assert list_distance(d) == d and (nbytes % 2048 or d % 2048 == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("numel,calls", [(21 * MB + 77, (1,)), (32 * MB, (1, 2)), (5 * MB + 1, (5, 1)), (300_001, (2,)), (257 * MB, (1,))])
def test_every_chunk_has_memory_of_its_own(numel, calls):
    """Lists long and short enough to share an allocation or not, appended in one call or several."""
    client = ps.PatrickStarClient(0, numel)
    params = [p for n in calls for p in client.append_flat_chunks(n)]
    if calls == (1, 2):
        params = params[1:]  # a parameter the optimizer is not given has no state chunks: its room stays unused
    opt = ps.FP16Adam(client, params, loss_scaler=ps.LossScaler(8.0), lr=1e-3)
    where = {p: [client.access_data(q) for q in (client.param_fp16_to_param_fp32_map[p], opt.state[p]["exp_avg"],
                                                 opt.state[p]["exp_avg_sq"], p)] for p in params}
    spans = sorted((t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for ts in where.values() for t in ts)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    for k, ts in enumerate(where.values()):
        for j, t in enumerate(ts):
            assert t.numel() == numel and t.data_ptr() % 1024 == 0 and int(torch.count_nonzero(t)) == 0
            t.fill_(1 + k * 4 + j)
    for k, ts in enumerate(where.values()):
        for j, t in enumerate(ts):
            assert bool((t == 1 + k * 4 + j).all())
    apart = [(a[1].data_ptr() - a[0].data_ptr()) % LIST_PERIOD for a in where.values()]
    if 80 * MB <= 4 * numel * calls[0] <= 1024 * MB and calls != (1, 2):
        assert LIST_CLEARANCE <= apart[0] <= LIST_PERIOD - LIST_CLEARANCE


@pytest.mark.gpu
@pytest.mark.parametrize("with_parameters", [False, True])
@pytest.mark.parametrize("chunk_type,dtype", [(ChunkType.MOMENTUM, torch.float), (ChunkType.VARIANCE, torch.float), (ChunkType.PARAM_FP32, torch.double)])
def test_lists_driven_on_their_own_get_memory_of_their_own(chunk_type, dtype, with_parameters):
    n = 24 * MB
    client = ps.PatrickStarClient(0, n)
    params = client.append_flat_chunks(1) if with_parameters else []
    p = torch.nn.Parameter(torch.tensor([], dtype=dtype), requires_grad=False)
    register_param(p, ParamType.CHUNK_BASED, dtype, "own")
    p.ps_attr.reset_shape(torch.Size([n]))
    client.append_tensor([p], dtype, AccessType.DATA, chunk_type)
    own = client.access_data(p)
    assert own.dtype == dtype and int(torch.count_nonzero(own)) == 0
    own.fill_(3)
    if params:
        opt = ps.FP16Adam(client, params, loss_scaler=ps.LossScaler(8.0), lr=1e-3)
        for q in (client.param_fp16_to_param_fp32_map[params[0]], opt.state[params[0]]["exp_avg"], opt.state[params[0]]["exp_avg_sq"], params[0]):
            t = client.access_data(q)
            assert t.numel() == n and int(torch.count_nonzero(t)) == 0
        opt.step()
        assert bool((own == 3).all())
