"""Gradients copied into their chunk slots many to a kernel: the entry point at the edges of its spans and batches, and
the engine's list of waiting gradients over the ways a backward pass can be run."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

import patrickstar_amd as ps
from patrickstar_amd import _lib

pytestmark = pytest.mark.gpu

# vectors of 8, spans of 2048 elements, 64 gradients to a launch
EDGES = [1, 7, 8, 9, 2040, 2041, 2047, 2048, 2049, 2056, 4096, 20001, 0, 768]


def _copy(grads, slots, state):
    rows = [(g.data_ptr() if g.numel() else None, s.data_ptr() if g.numel() else None, g.numel(), g.dtype == torch.half) for g, s in zip(grads, slots)]
    _lib.check(_lib.load().ps_grads_to_chunks((_lib.ps_grad_copy * len(rows))(*rows), len(rows), state, _lib.current_stream_handle()),
               "ps_grads_to_chunks")


@pytest.mark.parametrize("count", [1, 15, 64, 65, 150])
@pytest.mark.parametrize("kind", ["half", "float", "both"])
def test_lists_of_gradients_land_in_adjacent_slots_and_nowhere_else(kind, count):
    sizes = [EDGES[(3 * i + count) % len(EDGES)] for i in range(count)]
    dtypes = [torch.half if kind == "half" or (kind == "both" and i % 2) else torch.float for i in range(count)]
    grads = []
    for i, (n, dt) in enumerate(zip(sizes, dtypes)):
        off = i % 9
        grads.append((torch.randn(n + 9, device="cuda") * 50).to(dt)[off : off + n])
    for start in (0, 1, 5):
        chunk = torch.full((sum(sizes) + 16,), 7.0, dtype=torch.half, device="cuda")
        want = chunk.clone()
        slots, at = [], start
        for n, g in zip(sizes, grads):
            slots.append(chunk[at : at + n])  # one slot right behind the other
            want[at : at + n].copy_(g)
            at += n
        scaler = ps.DynamicLossScaler(init_scale=2**4)
        _copy(grads, slots, scaler.state_ptr)
        assert torch.equal(chunk.view(torch.int16), want.view(torch.int16))
        assert scaler.overflow_flag is False
    for i in {0, count // 2, count - 1}:
        for at in {0, sizes[i] // 2, sizes[i] - 1} if sizes[i] else ():
            keep = grads[i][at].clone()
            grads[i][at] = float("nan") if at else float("inf")
            scaler = ps.DynamicLossScaler(init_scale=2**4)
            _copy(grads, slots, scaler.state_ptr)
            assert scaler.overflow_flag is True, (i, at)
            _copy(grads, slots, None)  # without a state: a plain copy
            grads[i][at] = keep


def test_a_gradient_longer_than_one_launch_can_take():
    """A launch's grid ends at 2^24 - 1 spans of 2048 elements: the rest of the gradient goes into the next one."""
    n = (2**24 - 1) * 2048 + 4099
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 5 * n:
        pytest.skip("two tensors of 64 GiB do not fit")
    grad = torch.zeros(n, dtype=torch.half, device="cuda")
    slot = torch.full((n + 3,), 7.0, dtype=torch.half, device="cuda")
    marks = [0, 6, 7, 8, n - 4100, n - 4099, n - 4098, n - 2051, n - 1]
    for i, at in enumerate(marks):
        grad[at] = i + 1.0
    scaler = ps.DynamicLossScaler(init_scale=2**4)
    _copy([grad], [slot[1 : 1 + n]], scaler.state_ptr)
    assert scaler.overflow_flag is False
    assert [float(slot[1 + at]) for at in marks] == [i + 1.0 for i in range(len(marks))]
    assert float(slot[0]) == 7.0 and slot[1 + n :].tolist() == [7.0, 7.0]
    held = sum(int(torch.count_nonzero(slot[lo : lo + 2**30])) for lo in range(0, n + 3, 2**30))
    assert held == len(marks) + 3  # every other element has been copied
    grad[n - 1] = float("inf")
    _copy([grad], [slot[1 : 1 + n]], scaler.state_ptr)
    assert scaler.overflow_flag is True
    del grad, slot
    torch.cuda.empty_cache()


class _Net(torch.nn.Module):
    def __init__(self, reentrant):
        super().__init__()
        self.layers = torch.nn.ModuleList([torch.nn.Linear(24, 24) for _ in range(45)])  # 90 tensors: two launches
        self.reentrant = reentrant

    def forward(self, x):
        for i, layer in enumerate(self.layers):
            f = lambda y, m=layer: torch.tanh(m(y)) + y
            x = checkpoint(f, x, use_reentrant=True) if self.reentrant and i % 3 == 1 else f(x)
        return x.float().pow(2).mean()


@pytest.mark.parametrize("how", ["engine", "plain backward", "nested passes", "side stream", "after a failed pass", "small bound"])
def test_every_gradient_is_in_its_slot_when_backward_returns(how, monkeypatch):
    torch.manual_seed(0)
    config = {
        "optimizer": {"type": "Adam", "params": {"lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8, "weight_decay": 0}},
        "fp16": {"enabled": True, "loss_scale": 64},
        "default_chunk_size": 4096,
    }
    engine, optimizer = ps.initialize_engine(model_func=lambda: _Net(how == "nested passes"), local_rank=0, config=config)
    if how == "small bound":
        monkeypatch.setattr(type(engine), "PENDING_ELEMENTS", 1000)
    params = list(engine.module.parameters())
    slots = [engine.client.access_data(p) for p in params]
    assert [engine.client.data_address(p) for p in params] == [s.data_ptr() for s in slots]
    x = torch.randn(8, 24, device="cuda").half().requires_grad_()
    engine.module.reentrant, nested = False, engine.module.reentrant
    expected = torch.autograd.grad(engine(x) * 64, params)  # no hooks fire for autograd.grad
    engine.module.reentrant = nested
    torch.cuda.synchronize()
    if how == "after a failed pass":
        def refuse(grad):
            raise ValueError("refused")

        y = x.detach().clone().requires_grad_()
        y.register_hook(refuse)  # the last gradient of the pass
        kept = [s.clone() for s in slots]
        with pytest.raises(ValueError):
            engine.backward(engine(y))
        for s, k in zip(slots, kept):
            s.copy_(k)
    if how == "side stream":
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            loss = engine(x)
        torch.cuda.current_stream().wait_stream(side)
        engine.backward(loss)
    elif how == "plain backward":
        (engine(x) * 64).backward()
    else:
        engine.backward(engine(x))
    got = [s.clone() for s in slots]  # on the caller's stream, with nothing waited for
    assert all(p.grad is None for p in params) and not engine._pending
    for k, (a, b) in enumerate(zip(got, expected)):
        assert torch.equal(a, b), k
    optimizer.step()
    assert torch.isfinite(engine(x))


@pytest.mark.parametrize("nested", [False, True])
def test_a_plain_backward_after_a_failed_pass(nested):
    """The failed pass leaves gradients that were never copied (45 layers, 90 of them, 64 to a launch): they stay out of the
    slots, which the next pass reads as weights, and out of the overflow flag."""
    torch.manual_seed(0)
    config = {
        "optimizer": {"type": "Adam", "params": {"lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8, "weight_decay": 0}},
        "fp16": {"enabled": True, "loss_scale": 0, "initial_scale_power": 6},
        "default_chunk_size": 4096,
    }
    engine, optimizer = ps.initialize_engine(model_func=lambda: _Net(False), local_rank=0, config=config)
    params = list(engine.module.parameters())
    slots = [engine.client.access_data(p) for p in params]
    x = torch.randn(8, 24, device="cuda").half().requires_grad_()
    expected = torch.autograd.grad(engine(x) * 64, params)
    kept = [s.clone() for s in slots]
    engine.module.reentrant = nested

    def refuse(grad):
        raise ValueError("refused")

    y = x.detach().clone().requires_grad_()
    y.register_hook(refuse)
    with pytest.raises(ValueError):
        (engine(y) * float("inf")).backward()
    for s, k in zip(slots, kept):
        s.copy_(k)
    optimizer.has_overflow = False
    (engine(x) * 64).backward()
    assert all(torch.equal(a, b) for a, b in zip(slots, expected))
    assert optimizer.has_overflow is False and not engine._pending


def test_gradients_of_ordinary_layers_wait_for_a_launch_they_share(monkeypatch):
    """None of them is held by anybody else."""
    def model():
        return torch.nn.Sequential(torch.nn.Embedding(50, 32), torch.nn.TransformerEncoderLayer(32, 2, 64, dropout=0.0, batch_first=True),
                                   torch.nn.LayerNorm(32), torch.nn.Linear(32, 32), torch.nn.Conv1d(7, 7, 3))

    config = {
        "optimizer": {"type": "Adam", "params": {"lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8, "weight_decay": 0}},
        "fp16": {"enabled": True, "loss_scale": 64},
        "default_chunk_size": 8192,
    }
    engine, optimizer = ps.initialize_engine(model_func=model, local_rank=0, config=config)
    flush, lists = engine._flush_gradients, []
    monkeypatch.setattr(engine, "_flush_gradients", lambda waiting: (lists.append(len(waiting.gradients)), flush(waiting))[1])
    engine.backward(engine(torch.randint(0, 50, (3, 7), device="cuda")).float().pow(2).mean())
    n = sum(1 for _ in engine.module.parameters())
    assert sorted(k for k in lists if k) == [n]
