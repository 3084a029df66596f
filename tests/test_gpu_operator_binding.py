"""adam_update through the binding and through its general path: the same bits, and calls that are not of the ordinary form are
left to the general path, which accepts or refuses them as always."""
import numpy as np
import pytest
import torch

from patrickstar_amd import _lib, adam_op

pytestmark = pytest.mark.gpu
OPT = 7801


@pytest.fixture
def operator():
    adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
    yield
    adam_op.destroy_adam(OPT)


def _tensors(n, half, offset=0):
    gen = torch.Generator(device="cuda").manual_seed(n)
    p, m, v = (torch.randn(n + offset, device="cuda", generator=gen)[offset:] for _ in range(3))
    g = torch.randn(n + offset, device="cuda", generator=gen)[offset:]
    return [p, g.half() if half else g, m, v.square_()]


def _args(tensors, **kw):
    a = dict(step=3, lr=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8, weight_decay=0.01, bias_correction=True, loss_scale=8.0)
    a.update(kw)
    return (OPT, a["step"], a["lr"], a["beta1"], a["beta2"], a["epsilon"], a["weight_decay"], a["bias_correction"], *tensors, a["loss_scale"])


@pytest.mark.parametrize("n", [0, 1, 767, 4096, 70001])
@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("kw", [{}, {"lr": 0, "loss_scale": -1}, {"lr": np.float64(1e-4), "bias_correction": False}, {"loss_scale": 1e60}])
def test_both_ways_leave_the_same_bits(operator, n, half, kw):
    a, b = _tensors(n, half, 3), _tensors(n, half, 3)
    assert _lib.load().adam_update(*_args(a, **kw)) == 0
    assert adam_op._update(*_args(b, **kw)) == 0
    for x, y in zip(a, b):
        assert torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8))


class Sub(torch.Tensor):
    pass


NOT_PLAIN = {
    "a float step": lambda t: _args(t, step=3.0),
    "a negative step": lambda t: _args(t, step=-1),
    "a numpy number": lambda t: _args(t, lr=np.float32(1e-3)),
    "a tensor for a number": lambda t: _args(t, loss_scale=torch.tensor(8.0)),
    "an int for a truth value": lambda t: _args(t, bias_correction=1),
    "a subclass": lambda t: _args([t[0].as_subclass(Sub), *t[1:]]),
    "a host tensor": lambda t: _args([t[0], t[1].cpu(), *t[2:]]),
    "two dimensions": lambda t: _args([t[0].view(2, -1), *t[1:]]),
    "a stride": lambda t: _args([t[0], t[1], torch.zeros(2 * t[0].numel(), device="cuda")[::2], t[3]]),
    "another length": lambda t: _args([t[0], t[1], t[2], t[3][:-1]]),
    "another type": lambda t: _args([t[0].double(), *t[1:]]),
    "bfloat16 gradients": lambda t: _args([t[0], t[1].bfloat16(), *t[2:]]),
    "a sparse tensor": lambda t: _args([t[0], t[1].to_sparse(), *t[2:]]),
    "no tensor": lambda t: _args([None, *t[1:]]),
}


@pytest.mark.parametrize("what", NOT_PLAIN)
def test_other_calls_are_left_to_the_general_path(operator, what):
    tensors = _tensors(512, False)
    before = [t.clone() for t in tensors]
    assert _lib.load().adam_update(*NOT_PLAIN[what](tensors)) is None
    assert all(torch.equal(a, b) for a, b in zip(tensors, before))


def test_an_unknown_operator_raises_and_the_current_stream_is_used(operator):
    t = _tensors(1 << 22, True)
    with pytest.raises(RuntimeError, match="optimizer id 12345 was never created"):
        adam_op.adam_update(12345, *_args(t)[1:])
    side, want = torch.cuda.Stream(), [x.clone() for x in t]
    adam_op._update(*_args(want))
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        adam_op.adam_update(*_args(t))
        done = torch.cuda.Event()
        done.record()
    assert not done.query()  # queued behind the work of its own stream, and nobody waited for it
    done.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(t, want))
