"""The native Adam operator under the names the reference imports it by.

``patrickstar/ops/fp16_cpu_adam.py:177-193`` loads a pybind module ``cpu_adam_op``
with ``create_adam``, ``adam_update`` and ``destroy_adam``
(``patrickstar/ops/csrc/adam/cpu_adam.cpp:751-756``).  These are the same three
functions with the same argument meaning, taking flat torch tensors; the
arithmetic runs on the GPU through ``ps_adam_create`` / ``ps_adam_update`` /
``ps_adam_destroy``.  Like the reference's, each returns 0; failures raise.
"""
import torch

from . import _lib

_FLOAT, _HALF = torch.float, torch.half


def create_adam(optimizer_id, alpha=1e-3, betta1=0.9, betta2=0.999, eps=1e-8, weight_decay=0.0, adamw_mode=True,
                should_log=False):
    _lib.check(
        _lib.load().ps_adam_create(optimizer_id, alpha, betta1, betta2, eps, weight_decay, int(bool(adamw_mode)),
                                   int(bool(should_log))),
        "create_adam",
    )
    return 0


def destroy_adam(optimizer_id):
    _lib.check(_lib.load().ps_adam_destroy(optimizer_id), "destroy_adam")
    return 0


def adam_update(optimizer_id, step, lr, beta1, beta2, epsilon, weight_decay, bias_correction, params, grads, exp_avg,
                exp_avg_sq, loss_scale):
    """One update of one flat tensor, in place on ``params``, ``exp_avg`` and ``exp_avg_sq``.

    ``params``, ``exp_avg``, ``exp_avg_sq``: 1-D contiguous float32 tensors on the GPU (the reference asserts
    CPU tensors here, ``fp16_cpu_adam.py:222-225``); ``grads``: float32 or float16, never written;
    ``loss_scale <= 0``: no unscale.
    """
    rc = _lib.load().adam_update(optimizer_id, step, lr, beta1, beta2, epsilon, weight_decay, bias_correction, params, grads,
                                 exp_avg, exp_avg_sq, loss_scale)
    if rc is None:
        rc = _update(optimizer_id, step, lr, beta1, beta2, epsilon, weight_decay, bias_correction, params, grads, exp_avg,
                     exp_avg_sq, loss_scale)
    if rc:
        _lib.check(rc, "adam_update")
    return 0


def _update(optimizer_id, step, lr, beta1, beta2, epsilon, weight_decay, bias_correction, params, grads, exp_avg, exp_avg_sq,
            loss_scale):
    """adam_update of calls that are not of the ordinary form (plain tensors and numbers, on the current device), or that it
    refuses."""
    n = params.numel()
    if not (
        params.is_cuda and grads.is_cuda and exp_avg.is_cuda and exp_avg_sq.is_cuda
        and params.dim() == 1 and grads.dim() == 1 and exp_avg.dim() == 1 and exp_avg_sq.dim() == 1
        and params.is_contiguous() and grads.is_contiguous() and exp_avg.is_contiguous() and exp_avg_sq.is_contiguous()
        and params.dtype is _FLOAT and exp_avg.dtype is _FLOAT and exp_avg_sq.dtype is _FLOAT
        and (grads.dtype is _FLOAT or grads.dtype is _HALF)
        and grads.numel() == n and exp_avg.numel() == n and exp_avg_sq.numel() == n
    ):
        _refuse(params, grads, exp_avg, exp_avg_sq)
    with _lib.on_device(params.device):
        return _lib.load().ps_adam_update(
            optimizer_id, int(step), lr, beta1, beta2, epsilon, weight_decay, 1 if bias_correction else 0,
            params.data_ptr(), grads.data_ptr(), 1 if grads.dtype is _HALF else 0, exp_avg.data_ptr(),
            exp_avg_sq.data_ptr(), n, float(loss_scale), None, _lib.raw_stream(params.device),
        )


def _refuse(params, grads, exp_avg, exp_avg_sq):
    """Say which of adam_update's demands its tensors do not meet."""
    for name, t in (("params", params), ("grads", grads), ("exp_avg", exp_avg), ("exp_avg_sq", exp_avg_sq)):
        if not t.is_cuda:
            raise RuntimeError(f"adam_update: {name} must be a GPU tensor (got {t.device})")
        if t.dim() != 1 or not t.is_contiguous():
            raise RuntimeError(f"adam_update: {name} must be flat and contiguous (call .view(-1))")
    if params.dtype != torch.float or exp_avg.dtype != torch.float or exp_avg_sq.dtype != torch.float:
        raise TypeError("adam_update: params, exp_avg and exp_avg_sq must be float32")
    if grads.dtype not in (torch.float, torch.half):
        raise TypeError(f"adam_update: grads must be float32 or float16, got {grads.dtype}")
    raise RuntimeError("adam_update: tensors differ in length")
