"""Parity of the backward products where their split over K or their whole
rounds do not come out even, against the row-chunked restatement on the same
GPU (tests/torch_reference.py; tolerances as in tests/parity.py):

* 12 tiles split in 21 parts (252 workgroups) with a short last part;
* one tile split in more than 64 parts;
* grad_W (3 M-tiles x 100 N-tiles) as 85 column tiles in one round and 15 more
  split over K; grad_hidden (13 x 20 tiles) as 19 column tiles and one more;
* the same products under a memory limit that leaves no room for partials:
  they run unsplit, at the same chunk plan.
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
