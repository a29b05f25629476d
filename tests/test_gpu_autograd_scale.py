"""The autograd op's backward: each gradient times the incoming one, in its
input's dtype, as multiplying and converting the loss's own float32 gradients
gives it, bit for bit; sizes that end inside a block and inside a vector, any
subset of the inputs, and a batch of incoming gradients (vmap), which takes
torch's operators."""
import pytest

import orda_hip as H
from orda_hip import LossOptions, Teacher
from orda_hip.autograd import distillation_loss_autograd

pytestmark = pytest.mark.gpu


def make(bt, h, v, dtype, sep):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(bt + h + v)
    rnd = lambda r, c, std=1.0: (torch.randn(r, c, generator=g, device="cuda") * std).to(dtype)
    y = torch.randint(0, v, (bt,), generator=g, device="cuda")
    t = {"s": rnd(bt, h), "w": rnd(v, h, 0.1), "th": rnd(bt, h)}
    if sep:
        t["tw"] = rnd(v, h, 0.1)
    return t, y


def teacher(t):
    return Teacher.Separate(t["th"], t["tw"]) if "tw" in t else Teacher.Tied(t["th"])


OPTS = LossOptions(kd_weight=0.4, temperature=1.5, teacher_ce_weight=1.0)
NAMES = {"s": "grad_student_hidden", "w": "grad_weight", "th": "grad_teacher_hidden",
         "tw": "grad_teacher_weight"}


@pytest.mark.parametrize("want", ["s", "w", "sw", "wt", "swt"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("bt,h,v,sep", [(1, 1, 3, False), (7, 5, 31, True), (64, 128, 1000, False),
                                        (33, 72, 777, True)])
def test_backward_scales_and_converts(bt, h, v, sep, dtype, want):
    import torch
    t, y = make(bt, h, v, getattr(torch, dtype), sep)
    ref = H.distillation_loss(t["s"], t["w"], y, teacher(t), OPTS)
    leaves = {k: x.requires_grad_(True) for k, x in t.items() if k[0] in want}
    loss, _ = distillation_loss_autograd(t["s"], t["w"], y, teacher(t), OPTS)
    grads = torch.autograd.grad(2.7 * loss, list(leaves.values()))
    k = torch.tensor(2.7, device="cuda")
    for (name, x), g in zip(leaves.items(), grads):
        assert g.dtype == x.dtype and g.shape == x.shape
        assert torch.equal(g, (getattr(ref, NAMES[name]) * k).to(x.dtype)), name


def test_batched_incoming_gradients():
    import torch
    t, y = make(16, 24, 100, torch.bfloat16, False)
    t["s"].requires_grad_(True)
    ref = H.distillation_loss(t["s"].detach(), t["w"], y, teacher(t), OPTS).grad_student_hidden
    loss, _ = distillation_loss_autograd(t["s"], t["w"], y, teacher(t), OPTS)
    k = torch.tensor([1.0, 3.0], device="cuda")
    g, = torch.autograd.grad(loss, [t["s"]], grad_outputs=k, is_grads_batched=True)
    assert torch.equal(g, (ref * k[:, None, None]).to(torch.bfloat16))


@pytest.mark.parametrize("default", ["meta", "cuda", "cpu"])
def test_default_device_does_not_matter(default):
    """The op's outputs are on its inputs' device under any default device."""
    import torch
    t, y = make(16, 24, 100, torch.float32, False)
    want = H.distillation_loss(t["s"], t["w"], y, teacher(t), OPTS)
    t["w"].requires_grad_(True)
    with torch.device(default):
        loss, terms = distillation_loss_autograd(t["s"], t["w"], y, teacher(t), OPTS)
        g, = torch.autograd.grad(loss, [t["w"]])
    assert loss.item() == want.loss
    assert terms.tolist() == [want.student_ce, want.teacher_ce, want.kl]
    assert torch.equal(g, want.grad_weight)
