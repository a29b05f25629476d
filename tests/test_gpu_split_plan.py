"""Parity of the backward products where their split over K or their whole
rounds do not come out even, against the row-chunked restatement on the same
GPU (tests/torch_reference.py; tolerances as in tests/parity.py):

* 12 tiles split in 21 parts (252 workgroups) with a short last part;
* one tile split in more than 64 parts;
* grad_W (3 M-tiles x 100 N-tiles) as 85 column tiles in one round and 15 more
  split over K; grad_hidden (13 x 20 tiles) as 19 column tiles and one more;
* the same products under a memory limit that leaves no room for all their
  partials: they take fewer parts, at the same chunk plan, and grad_hidden of
  few tiles is not left on a few CUs.
"""
import pytest

from parity import check_grad_device, check_scalar
from torch_reference import loss_chunked

import orda_hip as H
from orda_hip import LossOptions, Teacher

pytestmark = pytest.mark.gpu

CASES = {
    "hidden-21-parts": (300, 768, 8001),
    "hidden-one-tile": (130, 200, 30011),
    "weight-column-tail": (2000, 768, 25600),
    "hidden-column-tail": (3300, 5120, 1500),
}


def inputs(torch, bt, h, v, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(bt + v)
    rnd = lambda r, c, std: (torch.randn(r, c, generator=g, device="cuda") * std).to(dtype)
    y = torch.randint(0, v, (bt,), generator=g, device="cuda")
    y[::11] = -100
    return rnd(bt, h, 1.0), rnd(v, h, h ** -0.5), y, rnd(bt, h, 1.0)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_uneven_splits(name, dtype):
    import torch
    torch.backends.cuda.matmul.allow_tf32 = False
    bt, h, v = CASES[name]
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    s, w, y, th = inputs(torch, bt, h, v, tdt)
    opts = LossOptions(kd_weight=0.5, temperature=1.5, label_smoothing=0.1)
    ref = loss_chunked(s, w, y, "tied", th, kd=0.5, T=1.5, alpha=0.1)
    free = H.Context(0)
    got = H.distillation_loss(s, w, y, Teacher.Tied(th), opts, ctx=free)
    held = free.workspace_bytes()
    free.close()
    tight = H.Context(0)
    tight.set_memory_limit(held - 4096)   # the last buffer to grow holds the partials
    small = H.distillation_loss(s, w, y, Teacher.Tied(th), opts, ctx=tight)
    assert tight.workspace_bytes() <= held - 4096
    tight.close()
    assert small.chunk_plan == got.chunk_plan
    for out in (got, small):
        for k in ("loss", "student_ce", "teacher_ce", "kl"):
            check_scalar(k, getattr(out, k), ref[k])
        for k in ("grad_student_hidden", "grad_weight", "grad_teacher_hidden"):
            check_grad_device(k, getattr(out, k), ref[k], dtype)


@pytest.mark.parametrize("short", [1 << 20, 12 << 20, 18 << 20])
def test_partials_that_do_not_fit_cost_no_idle_chip(short):
    """grad_hidden at 300 x 768 x 50257 is 6 to 12 tiles over a K of 50257: with
    K split over the CUs some 0.1 ms, unsplit ten times that. Under a limit
    that leaves too little room for its partials (18 MB) the product runs in
    the parts that fit, or the call makes room as it does for any other buffer;
    bound: three times the unbounded call's time of that product."""
    import torch
    s, w, y, _ = inputs(torch, 300, 768, 50257, torch.bfloat16)
    opts = LossOptions()

    def run(ctx):
        got = None
        for i in range(4):
            if i == 1:
                ctx.set_timing(True)
                ctx.reset_timing()
            got = H.distillation_loss(s, w, y, Teacher.Tied(s), opts, ctx=ctx)
        return got, ctx.kernel_time("gemm_grad_hidden")[0] / 3

    free = H.Context(0)
    want, t_free = run(free)
    limit = free.workspace_bytes() - short
    free.close()
    ctx = H.Context(0)
    ctx.set_memory_limit(limit)
    got, t = run(ctx)
    assert ctx.workspace_bytes() <= limit
    ctx.close()
    check_grad_device("grad_student_hidden", got.grad_student_hidden, want.grad_student_hidden, "bf16")
    check_grad_device("grad_weight", got.grad_weight, want.grad_weight, "bf16")
    assert t <= 3 * t_free
