"""torch autograd op over the fused distillation loss.

The reference's `distillation_loss` is the Rust analogue of upstream
`api.py::distillation_loss` together with the `DistillCEFunction`
forward/backward (src/api.rs:1-12). This module is that caller for torch: the
forward runs the whole fused loss on the GPU (liborda_hip.so through the C ABI,
which computes every gradient in the same call, src/api.rs:263-399) and keeps
the gradients; the backward scales them by the incoming gradient of the loss.

Gradients follow the reference (src/api.rs:244-258, 346-375): the KL term is
teacher-detached; the teacher's hidden rows (Tied, Separate) and the teacher's
weight (Separate) receive the teacher-CE gradient only when the teacher-CE
weight is positive; Precomputed teacher logits receive none. Each gradient is
returned in its input's dtype.
"""
from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch

from . import Context, distillation_loss
from . import _lib as L
from .types import LossOptions, OrdaError, Teacher, TeacherMode


def _plain(t):
    """A CUDA tensor with memory of its own (not one batched by vmap, as
    torch.autograd.grad's is_grads_batched makes, nor another wrapper)."""
    try:
        return t.is_cuda and type(t) is torch.Tensor and (t.data_ptr() != 0 or t.numel() == 0)
    except RuntimeError:
        return False


def _scaled(grads, dtypes, g_loss):
    """[g_loss * g as dtype] on the current stream, in one launch
    (orda_scale_gradients); a float32 gradient is scaled in place."""
    dev = grads[0].device
    out, parts = [], (L.ScaledGradient * len(grads))()
    scale = g_loss.to(torch.float32)
    p = scale.data_ptr()
    for part, g, dt in zip(parts, grads, dtypes):
        d = g if dt == torch.float32 else torch.empty_like(g, dtype=dt)
        part.src, part.dst, part.n = g.data_ptr(), d.data_ptr(), g.numel()
        part.dst_dtype = L.F32 if dt == torch.float32 else L.BF16
        out.append(d)
    err = ctypes.create_string_buffer(512)
    rc = L.load().orda_scale_gradients(dev.index or 0, torch.cuda.current_stream(dev).cuda_stream, p,
                                       parts, len(grads), err, 512)
    if rc != L.ORDA_OK:
        raise OrdaError(err.value.decode(), rc)
    return out


class DistillCEFunction(torch.autograd.Function):
    """loss, (student_ce, teacher_ce, kl) = DistillCEFunction.apply(
    student_hidden, weight, teacher_hidden, teacher_weight, labels,
    teacher_logits, mode, opts, lib_ctx)."""

    @staticmethod
    def forward(fctx, student_hidden, weight, teacher_hidden, teacher_weight, labels, teacher_logits,
                mode, opts, lib_ctx):
        teacher = Teacher(mode, hidden=None if teacher_hidden is None else teacher_hidden.detach(),
                          weight=None if teacher_weight is None else teacher_weight.detach(),
                          logits=None if teacher_logits is None else teacher_logits.detach())
        out = distillation_loss(student_hidden.detach(), weight.detach(), labels, teacher, opts,
                                ctx=lib_ctx)
        fctx.grads = (out.grad_student_hidden, out.grad_weight, out.grad_teacher_hidden,
                      out.grad_teacher_weight)
        fctx.dtypes = tuple(None if t is None else t.dtype
                            for t in (student_hidden, weight, teacher_hidden, teacher_weight))
        fctx.chunk_plan = out.chunk_plan
        dev = student_hidden.device
        # neither waits for the device: a fill, and a copy from pinned memory (of
        # the host, whatever torch's default device is)
        loss = torch.full((), out.loss, dtype=torch.float32, device=dev)
        comps = torch.tensor([out.student_ce, out.teacher_ce, out.kl], dtype=torch.float32,
                             device="cpu", pin_memory=dev.type == "cuda").to(dev, non_blocking=True)
        fctx.mark_non_differentiable(comps)
        return loss, comps

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(fctx, g_loss, g_comps):
        res = [None] * 4
        want = [i for i, (g, dt) in enumerate(zip(fctx.grads, fctx.dtypes))
                if g is not None and dt is not None and fctx.needs_input_grad[i]]
        if want:
            grads, dtypes = [fctx.grads[i] for i in want], [fctx.dtypes[i] for i in want]
            if _plain(g_loss) and all(_plain(g) and g.is_contiguous() for g in grads):
                scaled = _scaled(grads, dtypes, g_loss)
            else:
                scaled = [(g * g_loss.to(g.dtype)).to(dt) for g, dt in zip(grads, dtypes)]
            for i, g in zip(want, scaled):
                res[i] = g
        fctx.grads = None
        return (*res, None, None, None, None, None)


def distillation_loss_autograd(student_hidden: torch.Tensor, weight: torch.Tensor, labels,
                               teacher: Teacher, opts: Optional[LossOptions] = None, *,
                               ctx: Optional[Context] = None
                               ) -> Tuple[torch.Tensor, torch.Tensor]:
    """Differentiable form of `distillation_loss` for a training step.

    Returns ``(loss, components)``: ``loss`` is a 0-dim float32 tensor whose
    backward delivers the reference's gradients (scaled by the incoming
    gradient) to ``student_hidden``, ``weight`` and, where the reference has
    them, the teacher's hidden rows and weight; ``components`` holds
    ``[student_ce, teacher_ce, kl]`` (weight-free, kl including T², as in
    the reference's output, src/api.rs:71-92) and is not differentiable.
    Inputs must be GPU tensors.
    """
    opts = opts or LossOptions()
    if not (hasattr(student_hidden, "is_cuda") and student_hidden.is_cuda):
        raise ValueError("distillation_loss_autograd needs GPU tensors")
    mode = teacher.mode()
    th = teacher.hidden if mode in (TeacherMode.Tied, TeacherMode.Separate) else None
    tw = teacher.weight if mode == TeacherMode.Separate else None
    tl = teacher.logits if mode == TeacherMode.Precomputed else None
    return DistillCEFunction.apply(student_hidden, weight, th, tw, labels, tl, mode, opts, ctx)
