"""Fused decoupled AdamW on the HIP kernel ``dmuon_adamw_tensors``.

``fused_adamw_`` updates one bucket of the reference's ``_adamw_update_batch``
(``dmuon/optim/muon.py:1857-1916``): tensors that share the post-increment step count, the
parameter dtype (which the ``exp_avg``/``exp_avg_sq`` state shares, ``zeros_like(param)``) and
the gradient dtype. The dozen ``torch._foreach`` passes of the reference become one pass over
HBM; the per-element arithmetic and its rounding points are the same (see ``adamw.hip``).
There is no CPU path: tensors must live on the GPU.
"""
from __future__ import annotations

from typing import Optional, Sequence

import torch
from torch import Tensor

from .. import _C

_device_index = Tensor.get_device          # -1 for a CPU tensor
_CODES = {torch.float32: _C.DTYPE_F32, torch.bfloat16: _C.DTYPE_BF16}


def adamw_scalars(step: int, lr: float, betas: tuple[float, float], weight_decay: float,
                  eps: float) -> dict:
    """The scalars of one step, derived in double exactly as the reference derives them."""
    beta1, beta2 = float(betas[0]), float(betas[1])
    bc1 = 1.0 - beta1 ** step
    bc2 = 1.0 - beta2 ** step
    return {
        "apply_wd": 1 if weight_decay > 0 else 0,
        "wd_scale": 1.0 - lr * weight_decay,
        "beta1": beta1, "alpha1": 1.0 - beta1,
        "beta2": beta2, "alpha2": 1.0 - beta2,
        "bc2_sqrt": bc2 ** 0.5,
        "eps": float(eps),
        "neg_step": -(lr / bc1),
    }


def fused_adamw_(params: Sequence[Tensor], grads: Sequence[Tensor], exp_avgs: Sequence[Tensor],
                 exp_avg_sqs: Sequence[Tensor], *, step: int, lr: float,
                 betas: tuple[float, float], weight_decay: float, eps: float,
                 publish: Optional[Sequence[Optional[Tensor]]] = None) -> None:
    """In-place AdamW step of one bucket (same step, param dtype and grad dtype).

    ``publish``: optional forward copies (one per param, or None) that receive the new param
    rounded to their dtype in the same pass -- the owner's master -> forward publish; all of
    them share one dtype. Raises ``ValueError`` for mismatched lists, shapes or dtypes and
    ``RuntimeError`` for tensors that are not on the GPU or not contiguous (gradients are made
    contiguous).
    """
    n = len(params)
    if not (len(grads) == len(exp_avgs) == len(exp_avg_sqs) == n):
        raise ValueError("fused_adamw_: params, grads, exp_avgs, exp_avg_sqs differ in length")
    if n == 0:
        return
    if step < 1:
        raise ValueError(f"fused_adamw_: step must be >= 1, got {step}")
    dev = params[0].device
    if dev.type != "cuda":
        raise RuntimeError("fused_adamw_: tensors must live on the GPU (HIP kernel only)")
    if torch.cuda.is_current_stream_capturing():
        # the bias correction follows the host step count: a replay would repeat a stale step
        raise RuntimeError("fused_adamw_ cannot be captured into a graph (host step count); step "
                           "AdamW-routed parameters eagerly")
    pdt, gdt = params[0].dtype, grads[0].dtype
    if pdt not in _CODES or gdt not in _CODES:
        raise ValueError(f"fused_adamw_: unsupported dtypes param {pdt}, grad {gdt}")
    # each property over all tensors at once: a Python loop over the tensors costs more than the
    # update of a model's norm vectors
    owned = [*params, *exp_avgs, *exp_avg_sqs]
    index = dev.index if dev.index is not None else params[0].get_device()
    if not all(map(index.__eq__, map(_device_index, [*owned, *grads]))):
        raise RuntimeError("fused_adamw_: all tensors must be on one device")
    if {t.dtype for t in owned} != {pdt} or {g.dtype for g in grads} != {gdt}:
        raise ValueError("fused_adamw_: a bucket shares one param/state dtype and one grad dtype")
    numels = list(map(Tensor.numel, params))
    if not all(list(map(Tensor.numel, ts)) == numels for ts in (grads, exp_avgs, exp_avg_sqs)):
        raise ValueError("fused_adamw_: param, grad and state sizes differ")
    if not all(map(Tensor.is_contiguous, owned)):
        raise RuntimeError("fused_adamw_: params and AdamW state must be contiguous")
    gs = grads
    if not all(map(Tensor.is_contiguous, grads)):
        gs = [g.contiguous() for g in grads]
    qdt = None
    if publish is not None:
        if len(publish) != n:
            raise ValueError("fused_adamw_: publish must list one tensor (or None) per param")
        for p, q in zip(params, publish):
            if q is None:
                continue
            if q.device != dev or q.dtype not in _CODES or not q.is_contiguous():
                raise ValueError("fused_adamw_: publish targets must be contiguous fp32/bf16 "
                                 "tensors on the params' device")
            if q.numel() != p.numel() or (qdt is not None and q.dtype != qdt):
                raise ValueError("fused_adamw_: publish targets must match the params in size "
                                 "and share one dtype")
            qdt = q.dtype
    pubs = [0] * n if qdt is None else [0 if q is None else q.data_ptr() for q in publish]
    table = (_C.c_i64 * (6 * n))()
    for k, ts in enumerate((params, gs, exp_avgs, exp_avg_sqs)):
        table[k::6] = list(map(Tensor.data_ptr, ts))
    table[4::6] = pubs
    table[5::6] = numels
    s = adamw_scalars(step, lr, betas, weight_decay, eps)
    stream = torch.cuda.current_stream(dev).cuda_stream
    _C.call("dmuon_adamw_tensors", table, n, _CODES[pdt], _CODES[gdt],
            0 if qdt is None else _CODES[qdt], s["apply_wd"], s["wd_scale"], s["beta1"],
            s["alpha1"], s["beta2"], s["alpha2"], s["bc2_sqrt"], s["eps"], s["neg_step"], stream)
