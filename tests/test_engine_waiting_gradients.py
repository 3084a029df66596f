"""The engine's lists of waiting gradients, on the CPU: the engine's own hooks and bookkeeping, with a stand-in for the
kernel that copies the gradients of a list into their chunk slots."""
import copy
import ctypes
import threading
import types

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import patrickstar_amd as ps
from patrickstar_amd import _lib, engine as engine_module


class _Net(torch.nn.Module):
    def __init__(self, n=5):
        super().__init__()
        self.layers = torch.nn.ModuleList([torch.nn.Linear(6, 6) for _ in range(n)])
        self.nested = ()

    def forward(self, x):
        for i, layer in enumerate(self.layers):
            f = lambda y, m=layer: torch.tanh(m(y)) + y
            x = checkpoint(f, x, use_reentrant=True) if i in self.nested else f(x)
        return x.float().pow(2).mean()


def _tensor_at(address, numel, half):
    """The elements at an address, as a tensor that shares them."""
    raw = (ctypes.c_int16 * numel).from_address(address) if half else (ctypes.c_float * numel).from_address(address)
    return torch.frombuffer(raw, dtype=torch.half if half else torch.float)


class _Library:
    """What the engine calls of the native library, on host memory."""

    def __init__(self):
        self.flag = False  # the sticky overflow flag
        self.launches = []  # gradients in each

    def ps_grads_to_chunks(self, copies, n, state, stream):
        self.launches.append(n)
        for c in copies[:n]:
            if c.numel:
                slot = _tensor_at(c.d_slot_fp16, c.numel, True)
                slot.copy_(_tensor_at(c.d_grad, c.numel, c.grad_is_half != 0))
                self.flag = self.flag or not bool(torch.isfinite(slot).all())
        return 0


@pytest.fixture
def host(monkeypatch):
    """(engine, params, slots, library): an engine over a net on the CPU."""
    library = _Library()
    native = _lib.load()
    monkeypatch.setattr(engine_module, "_lib", types.SimpleNamespace(
        load=lambda: library, check=_lib.check, ps_grad_copy=_lib.ps_grad_copy, raw_stream=lambda device: 0, on_device=lambda device: _lib._NO_GUARD,
    ))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: types.SimpleNamespace(cuda_stream=0))
    assert native is not library
    torch.manual_seed(0)
    config = {"optimizer": {"type": "Adam", "params": {"lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8, "weight_decay": 0}},
              "fp16": {"enabled": True, "loss_scale": 64}}
    client = ps.PatrickStarClient(0, 512, device="cpu")
    model = client.register_model(_Net())
    engine = ps.PatrickStarEngine(model=model, client=client, config=config)
    params = list(engine.module.parameters())
    return engine, params, [client.access_data(p) for p in params], library


def _expected(engine, x, params):
    nested, engine.module.nested = engine.module.nested, ()
    want = torch.autograd.grad(engine(x) * 64, params)  # no hooks fire for autograd.grad
    engine.module.nested = nested
    return want


def _input(seed=1):
    return torch.randn(3, 6, generator=torch.Generator().manual_seed(seed)).half().requires_grad_()


def _same(slots, want):
    return [bool(torch.equal(s.view(w.shape), w)) for s, w in zip(slots, want)]


class _Refused(Exception):
    pass


def _failing_pass(engine, x, start, inf=False):
    """A backward pass that raises after every parameter's hook has run (``start`` begins it)."""
    y = x.detach().clone().requires_grad_()

    def refuse(grad):
        raise _Refused

    y.register_hook(refuse)  # the last gradient of the pass
    with pytest.raises(_Refused):
        start(engine(y) * (float("inf") if inf else 64))


# 1: a copy for every gradient; 3: some copied, some waiting; 64: all of them waiting when the pass fails
@pytest.mark.parametrize("at_once", [1, 3, 64])
@pytest.mark.parametrize("nested", [(), (1, 2), (0, 3)])
@pytest.mark.parametrize("retry", ["plain backward", "engine"])
def test_gradients_of_a_failed_pass_stay_out_of_the_next_one(host, monkeypatch, at_once, nested, retry):
    engine, params, slots, library = host
    monkeypatch.setattr(type(engine), "PENDING_GRADIENTS", at_once)
    x = _input()
    engine.module.nested = nested
    kept = [s.clone() for s in slots]
    want = _expected(engine, x, params)
    _failing_pass(engine, _input(2), lambda loss: loss.backward(), inf=True)
    assert not engine._pending
    library.flag = False  # the caller clears the flag and restores the parameters
    for s, k in zip(slots, kept):
        s.copy_(k)
    if retry == "engine":
        engine.backward(engine(x))
    else:
        (engine(x) * 64).backward()
    assert all(_same(slots, want))
    assert not library.flag and not engine._pending and all(p.grad is None for p in params)


@pytest.mark.parametrize("nested", [(1, 2), (0, 3), (4,), (0, 1, 2, 3, 4)])
def test_a_nested_pass_leaves_the_outer_list_waiting(host, nested):
    engine, params, slots, library = host
    engine.module.nested = nested
    x = _input()
    want = _expected(engine, x, params)
    engine.backward(engine(x))
    assert all(_same(slots, want)) and not engine._pending
    # one copy at the end of each nested pass, one at the end of the outer one if it had gradients of its own
    assert len(library.launches) == len(nested) + (len(nested) < len(engine.module.layers))


def test_two_failed_passes_and_a_failed_nested_one(host):
    engine, params, slots, library = host
    x = _input()
    kept = [s.clone() for s in slots]
    want = _expected(engine, x, params)
    engine.module.nested = (0, 1)

    def refuse(grad):
        raise _Refused

    for _ in range(2):
        handle = engine.module.layers[0].weight.register_hook(refuse)  # raises inside the nested pass over layer 0
        with pytest.raises(_Refused):
            engine.backward(engine(x))
        handle.remove()
        assert not engine._pending
        for s, k in zip(slots, kept):
            s.copy_(k)
        for p in params:
            p.grad = None
    (engine(x) * 64).backward()
    assert all(_same(slots, want)) and not engine._pending


@pytest.mark.parametrize("inf_in_first", [False, True])
def test_a_parameter_of_two_passes_keeps_the_later_gradient(host, inf_in_first):
    """A layer outside a nested pass (its gradient comes first, and waits) and inside it: two gradients for one slot."""
    engine, params, slots, library = host
    first = engine.module.layers[0]
    twin = copy.deepcopy(first)

    def forward(x, inner):
        f = lambda y: torch.tanh(engine.module.layers[1](inner(y)))
        x = checkpoint(f, x, use_reentrant=True) if inner is first else f(x)
        x = torch.tanh(first(engine.module.layers[2](x)))
        return x.float().pow(2).mean() * 64

    x = _input()
    want = torch.autograd.grad(forward(x, twin), list(twin.parameters()))
    if inf_in_first:
        first.weight.register_hook(lambda g: g * float("inf") if not library.launches and not seen.append(1) else g)
    seen = []
    forward(x, first).backward()
    assert bool(seen) == inf_in_first == library.flag and not engine._pending
    if not inf_in_first:
        assert all(_same(slots[:2], want))


def test_passes_of_two_threads_keep_their_gradients_apart(host):
    engine, params, slots, library = host
    x = _input()
    halves = [engine.module.layers[:2], engine.module.layers[2:]]
    want, losses = [], []
    for layers in halves:
        y = x
        for layer in layers:
            y = torch.tanh(layer(y))
        losses.append(y.float().pow(2).mean() * 64)
        want += torch.autograd.grad(losses[-1], [p for layer in layers for p in layer.parameters()], retain_graph=True)
    both = threading.Barrier(2)
    for i, layers in enumerate(halves):
        layers[0].weight.register_hook(lambda g: (both.wait(30), None)[1])  # neither pass ends before the other's last gradient
    errors = []

    def run(loss):
        try:
            loss.backward()
        except Exception as e:
            errors.append(e)

    workers = [threading.Thread(target=run, args=(loss,)) for loss in losses]
    for w in workers:
        w.start()
    for w in workers:
        w.join(60)
    assert not errors and all(_same(slots, want)) and not engine._pending


def _readers(engine, params):
    """What a program may do in the middle of a backward pass to see the gradients that are complete."""
    client, optimizer = engine.client, engine.optimizer
    optimizer._plan, optimizer._trainable_seen = {"kind": "empty"}, tuple(p.requires_grad for p in optimizer.param_groups[0]["params"])
    return {
        "access_data": lambda p: client.access_data(p),
        "settle all": lambda p: client.settle_gradients(),
        "settle one": lambda p: client.settle_gradients(p),
        "has_overflow": lambda p: optimizer.has_overflow,
        "clear the flag": lambda p: setattr(optimizer, "has_overflow", False),
        "reset": lambda p: optimizer.has_overflow_and_reset_param(),
        "step": lambda p: optimizer.step(),
    }


@pytest.mark.parametrize("how", ["access_data", "settle all", "settle one", "has_overflow", "clear the flag", "reset", "step"])
def test_a_complete_gradient_is_in_its_slot_for_whoever_looks_during_backward(host, how):
    engine, params, slots, library = host
    x = _input()
    want = _expected(engine, x, params)
    look, seen = _readers(engine, params)[how], []

    def hook(p):
        i = [q is p for q in params].index(True)
        look(p)
        seen.append((i, slots[i].clone()))

    for p in params:
        p.register_post_accumulate_grad_hook(hook)  # behind the engine's own
    engine.backward(engine(x))
    assert sorted(i for i, _ in seen) == list(range(len(params)))
    assert all(torch.equal(s.view(want[i].shape), want[i]) for i, s in seen)


@pytest.mark.parametrize("how", ["access_data", "step"])
def test_gradients_are_in_their_slots_for_a_callback_that_runs_before_the_engines(host, how):
    engine, params, slots, library = host
    x = _input()
    want = _expected(engine, x, params)
    look, seen = _readers(engine, params)[how], []

    def at_end():
        for p in params:
            look(p)
        seen.extend(s.clone() for s in slots)

    loss = engine(x) * 64
    loss.register_hook(lambda g: torch.autograd.Variable._execution_engine.queue_callback(at_end))
    loss.backward()
    assert len(seen) == len(params) and all(_same(seen, want)) and not engine._pending


def test_a_dynamic_scaler_asks_for_waiting_gradients_before_its_flag_is_read():
    scaler, asked = ps.DynamicLossScaler(), []
    scaler.before_flag = lambda: asked.append(1)
    assert scaler.overflow_flag is False and asked == [1]
    scaler.materialize = lambda: (_ for _ in ()).throw(_Refused())
    with pytest.raises(_Refused):
        scaler.update_scale(None)
    assert asked == [1, 1]


class _Product(torch.autograd.Function):
    """x @ w.T whose weight gradient is formed in a workspace that every call uses again."""

    @staticmethod
    def forward(ctx, x, w, workspace):
        ctx.save_for_backward(x, w)
        ctx.workspace = workspace
        return x @ w.t()

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        torch.mm(g.t(), x, out=ctx.workspace.view(w.shape))
        return g @ w, ctx.workspace.view(w.shape), None


@pytest.mark.parametrize("how", ["workspace", "pieces of one tensor", "kept by a hook"])
def test_a_gradient_in_memory_that_others_hold_is_copied_before_they_use_it_again(host, how):
    engine, params, slots, library = host
    weights = [layer.weight for layer in engine.module.layers]
    workspace = torch.zeros(36, dtype=torch.half)
    x = _input()

    def forward(product):
        y = x
        for w in weights:
            y = torch.tanh(product(y, w)) + y
        return y.float().pow(2).mean() * 64

    want = torch.autograd.grad(forward(lambda y, w: y @ w.t()), weights)
    if how == "workspace":
        forward(lambda y, w: _Product.apply(y, w, workspace)).backward()
    elif how == "kept by a hook":
        kept = []
        for w in weights:
            ready, w._post_accumulate_grad_hooks = w._post_accumulate_grad_hooks, None
            w.register_post_accumulate_grad_hook(lambda p: kept.append(p.grad))  # in front of the engine's
            for hook in ready.values():
                w.register_post_accumulate_grad_hook(hook)
        weights[0].register_post_accumulate_grad_hook(lambda p: ([g.zero_() for g in kept], None)[1])
        forward(lambda y, w: y @ w.t()).backward()
    else:
        whole = torch.zeros(len(weights), 6, 6, dtype=torch.half)
        for w, piece in zip(weights, whole):
            w.grad = piece  # accumulated into, in place
        # once the last gradient is complete, and before the pass ends, their owner clears the tensor for the next pass
        weights[0].register_post_accumulate_grad_hook(lambda p: (whole.zero_(), None)[1])
        forward(lambda y, w: y @ w.t()).backward()
    got = [engine.client.access_data(w) for w in weights]
    assert all(_same(got, want))


def test_ordinary_gradients_share_a_launch(host):
    engine, params, slots, library = host
    engine.backward(engine(_input()))
    assert library.launches == [len(params)]


def test_a_gradient_accumulated_outside_any_backward_pass_is_copied_at_once(host):
    engine, params, slots, library = host
    for p, slot in zip(params, slots):
        accumulate = p.view_as(p).grad_fn.next_functions[0][0]
        g = torch.randn(p.shape).half()
        accumulate(g.clone())
        assert torch.equal(slot, g) and p.grad is None
    assert not engine._pending
