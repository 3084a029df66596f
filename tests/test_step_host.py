"""The short ways of ``FP16Adam.step`` on the host: torch's wrapper around a step is left out only where nobody would notice, and a
plan whose numbers are read by the binding is the plan that a look at every parameter makes."""
import random
import types
from fractions import Fraction

import numpy as np
import pytest
import torch
from torch.optim.optimizer import register_optimizer_step_post_hook, register_optimizer_step_pre_hook

import patrickstar_amd as ps
from patrickstar_amd import _lib
from test_host_logic import _device_decided_step_on_the_cpu, _tiny_optimizer


def _compiled():
    """Takes every step for one that it cannot do at once."""
    compiled = getattr(_lib.load(), "compiled", None)
    if compiled is None:
        pytest.skip("without the binding there is only the long way")
    return types.SimpleNamespace(quiet=compiled.quiet, same_flags=lambda params, flags: False)


@pytest.fixture
def optimizer(monkeypatch):
    compiled = _compiled()
    optimizer, library = _device_decided_step_on_the_cpu(monkeypatch, ps.DynamicLossScaler())
    library.compiled = compiled
    return optimizer


def _ranges(profile):
    return [e.name for e in profile.events() if e.name.startswith("Optimizer.step#")]


def test_hooks_and_profilers_see_every_step(optimizer):
    seen = []
    handles = [optimizer.register_step_pre_hook(lambda *a: seen.append("before")), optimizer.register_step_post_hook(lambda *a: seen.append("behind"))]
    optimizer.step()
    assert seen == ["before", "behind"]
    for h in handles:
        h.remove()
    optimizer.step()
    assert seen == ["before", "behind"]
    for register in (register_optimizer_step_pre_hook, register_optimizer_step_post_hook):
        handle = register(lambda *a: seen.append("every"))
        optimizer.step()
        handle.remove()
    assert seen[2:] == ["every", "every"]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        optimizer.step()
    assert _ranges(profile) == ["Optimizer.step#FP16Adam.step"]
    assert len(optimizer._lib.names) == 5


def test_a_schedulers_wrapper_and_a_subclass_are_gone_through(monkeypatch):
    class Sub(ps.FP16Adam):
        def step(self, closure=None):
            seen.append("sub")
            return super().step(closure)

    seen = []
    compiled = _compiled()
    optimizer, library = _device_decided_step_on_the_cpu(monkeypatch, ps.DynamicLossScaler(), Sub)
    library.compiled = compiled
    optimizer.register_step_pre_hook(lambda *a: seen.append("hook"))
    torch.optim.lr_scheduler.LambdaLR(optimizer, lambda k: 1.0)
    optimizer.step()
    assert seen == ["hook", "sub"] and len(library.names) == 1
    assert optimizer.step(lambda: 3.0) == 3.0


VALUES = [1e-3, 0.5, 0, 1, np.float64(0.25), float("nan"), float("inf")]
OTHERS = [Fraction(1, 8), np.float32(0.125), True, torch.tensor(0.75)]  # numbers, but not of the ordinary form


@pytest.mark.parametrize("seed", range(6))
def test_numbers_read_by_the_binding_make_the_same_plan(seed, monkeypatch):
    _compiled()
    rng = random.Random(seed)
    _, model, a = _tiny_optimizer()
    _, _, b = _tiny_optimizer()
    both = [(o, list(o.param_groups[0]["params"])) for o in (a, b)]
    count = len(both[0][1])
    again = []
    plan_again = ps.FP16Adam._plan_again
    monkeypatch.setattr(ps.FP16Adam, "_plan_again", lambda self, *args: again.append(plan_again(self, *args)) or again[-1])

    def write(i, key, value):
        for o, params in both:
            o.state[params[i]][key] = value

    other = None
    for _ in range(60):
        if other is not None:
            for i in range(count):
                write(i, other, 0.125)
            other = None
        what = rng.randrange(6)
        if what == 0:
            i, on = rng.randrange(count), rng.random() < 0.7
            for _, params in both:
                params[i].requires_grad_(on)
        elif what == 1:
            write(rng.randrange(count), "step", rng.randrange(3))
        elif what == 2:
            key, value = rng.choice(["lr", "eps", "weight_decay"]), rng.choice(VALUES + OTHERS)
            other = key
            for i in range(count):
                write(i, key, value)
        elif what == 3:
            write(rng.randrange(count), "betas", rng.choice([(0.9, 0.999), [0.5, 0.25], (0, 1e-3)]))
        else:
            write(rng.randrange(count), rng.choice(["lr", "eps", "weight_decay"]), rng.choice(VALUES[:5]))
        a._make_plan()
        b._numbers = None  # looks at every parameter
        b._make_plan()
        assert a._plan["kind"] == b._plan["kind"] and a._common_step == b._common_step
        if a._plan["kind"] == "uniform":
            assert a._plan["hyper"] == b._plan["hyper"]
        if a._plan["kind"] != "each":
            continue
        tables = []
        for o, _ in both:
            monkeypatch.setattr(o, "_tensor_rows", lambda trainable: (None, None, len(trainable)))
            o._each_static = None if o is b else o._each_static
            tables.append(o._each_table(o._plan))
        (_, _, n, x, _, *rest_a), (_, _, m, y, _, *rest_b) = tables
        assert n == m and rest_a == rest_b
        if a._numbers is not None and x is a._numbers.each:
            a._lib.compiled.write_steps(a._numbers.at, n, 7, a._numbers.distances_at)
            assert [x[i].step - 7 for i in range(n)] == rest_a[1]
        for i in range(n):
            x[i].step = y[i].step = 0
        assert bytes(x) == bytes(y)
    assert True in again and False in again


def test_a_plan_whose_numbers_were_read_by_the_binding_outlives_new_payloads(monkeypatch):
    _compiled()
    _, _, optimizer = _tiny_optimizer()
    params = list(optimizer.param_groups[0]["params"])
    monkeypatch.setattr(optimizer, "_tensor_rows", lambda trainable: (None, None, len(trainable)))
    for k in range(4):
        for i, p in enumerate(params):
            optimizer.state[p]["lr"] = 0.5 ** (k + i)
        optimizer._make_plan()
    assert optimizer._plan["kind"] == "each" and optimizer._plan["entries"] is None
    optimizer.invalidate_tables()
    each = optimizer._each_table(optimizer._plan or optimizer._make_plan())[3]
    assert [e.lr for e in each] == [0.5 ** (3 + i) for i in range(len(params))]
