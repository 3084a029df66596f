"""A device-decided step with per-tensor numbers as one call (the probe forms the constants, the first launch of the update replaces
the state), against the probe, the step and the scale update as calls of their own: payloads, step state and log the same bits.  One launch
and several, lists that are probed in chunks of several lengths, both sides of the lines, overflows on steps next to one another."""
import ctypes

import pytest
import torch

from patrickstar_amd import DynamicLossScaler, FP16Adam, PatrickStarClient, _lib, adam_op
from test_gpu_near_tensor_lists import SHAPES, Lists

pytestmark = pytest.mark.gpu
OPT = 8401


class _Each:
    def __init__(self, way, sizes, gap, moved, classes, arithmetics, decays, chunks):
        self.way, self.opt, self.lists = way, OPT + way, Lists(sizes, gap, moved, 2.0**12, seed=len(sizes) + gap)
        adam_op.create_adam(self.opt, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
        self.scaler = DynamicLossScaler(init_scale=2.0**12, scale_window=3).materialize("cuda:0", betas=(0.9, 0.999))
        self.scaler.enable_log(16)
        n = self.lists.n
        self.each = (_lib.ps_tensor_call * n)()
        for i in range(n):
            self.each[i] = _lib.ps_tensor_call(1e-3 * 0.9 ** (i % classes), 0.9, 0.999, 1e-8, 0.01 * (i % decays != 1), i % 2, i % 2 if arithmetics == 2 else -1, 0)
        self.calls = sum(e.arithmetic != _lib.PS_ARITH_TORCH for e in self.each)
        self.work = torch.empty(_lib.load().ps_tensors_each_workspace_bytes(n), dtype=torch.uint8, device="cuda")
        # what is probed: the fp16 list in chunks, the last one shorter
        h = self.lists.data[3]
        length = (h.numel() + chunks - 1) // chunks // 8 * 8 + 8
        used = [max(0, min(length, h.numel() - k * length)) for k in range(chunks)]
        self.probed = _lib.chunk_array([[t[min(k * length, h.numel() - 1) :].data_ptr() for t in self.lists.data] for k in range(chunks)])
        self.chunks, self.length, self.used = chunks, length, _lib.size_array(used)

    def step(self):
        lib, s, x = _lib.load(), _lib.current_stream_handle(), self.lists
        probed = (self.probed, self.chunks, self.length, self.used)
        if self.way == 0:
            _lib.check(lib.ps_overflow_scan_chunks(*probed, self.scaler.state_ptr, s), "probe")
            _lib.check(lib.ps_adam_step_tensors_each(self.opt, 1, x.rows, x.numels, self.each, x.n, -1.0, self.scaler.state_ptr,
                                                     self.work.data_ptr(), self.work.numel(), s), "step")
            self.scaler.update_scale(None, operator_calls=self.calls)
            return
        scratch = self.scaler._scratch.data_ptr() if self.way == 1 else None
        _lib.check(lib.ps_adam_step_tensors_dynamic(self.opt, 1, *probed, x.rows, x.numels, self.each, x.n, self.scaler.state_ptr,
                                                    *self.scaler.log_arguments(), self.calls, self.work.data_ptr(), self.work.numel(), scratch,
                                                    _lib.PS_STEP_SCRATCH_BYTES if scratch else 0, s), "at once")


def _compare(runs, k):
    for r in runs[1:]:
        for name, x, y in zip(("p", "m", "v", "h"), runs[0].lists.whole(), r.lists.whole()):
            ints = torch.int16 if x.dtype == torch.half else torch.int32
            assert torch.equal(x.view(ints), y.view(ints)), (k, r.way, name)
        assert torch.equal(runs[0].scaler._state, r.scaler._state), (k, r.way)
        assert torch.equal(runs[0].scaler._log, r.scaler._log), (k, r.way)


@pytest.mark.parametrize("shape,gap,moved,classes,arithmetics,decays,chunks", [
    ("one", 0, False, 1, 1, 1, 1), ("equal_lengths", 0, False, 5, 1, 1, 3), ("short", 1, False, 24, 1, 1, 2), ("short", 1, False, 25, 1, 1, 2),
    ("ends_of_segments", 4, False, 3, 2, 3, 64), ("ten_segments", 0, False, 2, 1, 2, 65), ("three_launches", 1, False, 7, 2, 3, 5),
    ("with_empty", 0, False, 3, 1, 1, 1), ("layer", 4, False, 12, 1, 2, 4), ("layer", 4, True, 12, 1, 2, 4), ("long", 0, False, 6, 1, 1, 2),
])
def test_at_once_is_the_three_calls(shape, gap, moved, classes, arithmetics, decays, chunks):
    sizes = [9 << 20, (9 << 20) - 7, 255, 3 << 20, 12 << 20, 1, 2 << 20] if shape == "long" else SHAPES[shape]
    runs = [_Each(way, sizes, gap, moved, classes, arithmetics, decays, chunks) for way in range(3)]
    n = runs[0].lists.data[3].numel()
    # where an overflow is, if there is one; whether the flag was raised before
    for k, (poison, flag) in enumerate([(None, 0), (0, 0), (n - 1, 0), (None, 0), (n // 2, 0), (None, 1), (None, 0), (None, 0)]):
        for r in runs:
            grads = r.lists.data[3]
            grads.copy_((r.lists.data[0] * 50).half())
            if poison is not None:
                grads[poison] = float("nan") if k % 2 else float("inf")
            if flag:
                r.scaler._state[_lib.ps_step_state.overflow.offset :][:4].view(torch.int32).fill_(1)
            r.step()
        _compare(runs, k)
        assert runs[1].scaler.last_step_skipped == (poison is not None or bool(flag)), k
    for r in runs:
        adam_op.destroy_adam(r.opt)


def test_it_shares_its_scratch_with_whole_list_steps_and_replays_in_a_graph():
    """A whole-list step in two launches between the replays: the words of the probe are taken in turn by both."""
    runs = [_Each(way, SHAPES["layer"], 0, False, 6, 1, 1, 1) for way in range(2)]
    stream = torch.cuda.Stream()

    def whole(r):
        scratch = r.scaler._scratch.data_ptr() if r.way else None
        _lib.check(_lib.load().ps_adam_step_chunks_dynamic_scratch(r.opt, 1e-3, 1e-8, 0.01, 1, r.probed, 1, r.lists.data[3].numel(), None, None, 1,
                                                                   r.scaler.state_ptr, *r.scaler.log_arguments(), 1, scratch,
                                                                   _lib.PS_STEP_SCRATCH_BYTES if scratch else 0, _lib.current_stream_handle()), "whole list")

    with torch.cuda.stream(stream):
        for r in runs:
            r.step()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            runs[1].step()
        for k in range(6):
            for r in runs:
                r.lists.data[3].copy_((r.lists.data[0] * 50).half())
                if k in (1, 2, 4):
                    r.lists.data[3][k * 1000] = float("inf")
                if k == 3:
                    whole(r)
            if k != 3:
                runs[0].step()
                graph.replay()
            stream.synchronize()
            _compare(runs, k)
    for r in runs:
        adam_op.destroy_adam(r.opt)


@pytest.mark.parametrize("arithmetic", ["operator", "torch"])
@pytest.mark.parametrize("schedule", [False, True])
def test_a_step_over_some_of_the_tensors_is_done_at_once(schedule, arithmetic, monkeypatch):
    """One set of numbers for all that is trainable; without scratch memory the optimizer takes the probe, the step and the scale update."""
    outs, states, calls = [], [], []
    for at_once in (True, False):
        torch.manual_seed(3)
        client = PatrickStarClient(0, 40000)
        with torch.device("cuda"):
            model = torch.nn.Sequential(*[torch.nn.Linear(97, 101), torch.nn.Linear(101, 64), torch.nn.LayerNorm(64), torch.nn.Linear(64, 300)])
        client.register_model(model)
        params = list(model.parameters())
        for p in params[:3]:
            p.requires_grad_(False)
        scaler = DynamicLossScaler(init_scale=2.0**10, scale_window=2)
        optimizer = FP16Adam(client, params, loss_scaler=scaler, lr=1e-3, weight_decay=0.01, use_adamw=True, arithmetic=arithmetic)
        if not at_once:
            scaler._scratch = None
        step_at_once = optimizer._step_each_at_once
        monkeypatch.setattr(optimizer, "_step_each_at_once", lambda *args: calls.append(step_at_once(*args)) or calls[-1])
        for k in range(8):
            for p in params[3:]:
                p.data.copy_(torch.linspace(-1, 1, p.numel(), device="cuda").view(p.shape) * (k + 1))
                if schedule:
                    optimizer.state[p]["lr"] = 1e-3 * 0.5**k
            if k in (2, 3, 6):
                params[4 if k == 3 else -1].data.view(-1)[0] = float("inf")
            if k == 5:
                params[3].requires_grad_(False)
            optimizer.step()
        outs.append([client.chunk_list[c].payload.clone() for pos in client.positions() for c in (pos.fp32, pos.exp_avg, pos.exp_avg_sq, pos.fp16)])
        state = scaler._read()
        # (the record of a step's last call, when pending_operator_step says that there is none)
        fields = [name for name, *_ in state._fields_ if not name.startswith(("reserved", "pending_beta", "pad", "_"))]
        states.append({name: getattr(state, name) for name in fields})
        assert scaler.skipped_steps == 3 and optimizer.state[params[4]]["step"] == 5
    assert calls == [True] * 8 + [False] * 8 and states[0] == states[1] and states[0]["pending_operator_step"] == 0
    for x, y in zip(*outs):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
