"""bf16 products on 128 x 256 tiles (logits and grad_W of short K or few tiles)
at the edges of their tiles and stages: rows around a tile and around the
paired blocks of 16, hidden widths that are not a multiple of the 32-element
stage or leave a single stage, odd vocabularies, K of one to a few stages, two
staging groups (the accumulating grad_W), each teacher mode; against the
row-chunked restatement on the same GPU (tolerances as in tests/parity.py).
Each case names the products that take these tiles, by the kernels it launches:
l logits, w grad_W; some keep to the 256 x 256 ones."""
import pytest

from helpers import kernels_of
from parity import check_grad_device, check_scalar
from torch_reference import loss_chunked

import orda_hip as H
from orda_hip import ChunkSize, LossOptions, Teacher

pytestmark = pytest.mark.gpu

CASES = [  # mode, bt, h, ht, v, groups, products
    ("tied", 1, 8, 8, 257, 1, "lw"), ("tied", 63, 24, 24, 1000, 1, "lw"), ("tied", 65, 72, 72, 255, 1, "lw"),
    ("tied", 127, 200, 200, 5003, 1, "lw"), ("tied", 129, 264, 264, 8191, 1, "lw"),
    ("tied", 300, 768, 768, 20001, 1, ""), ("tied", 300, 768, 768, 50257, 1, "lw"),
    ("tied", 1000, 256, 256, 8000, 4, "lw"),
    ("none", 128, 40, 40, 513, 1, "lw"), ("none", 257, 96, 96, 3000, 2, "lw"),
    ("none", 1900, 768, 768, 12345, 1, ""), ("none", 1900, 512, 512, 12345, 1, "lw"),
    ("none", 1300, 256, 256, 30011, 1, "w"),
    ("separate", 130, 136, 72, 4001, 1, "lw"), ("separate", 600, 256, 512, 9000, 3, "lw"),
    ("precomputed", 140, 160, 0, 4008, 2, "w"),
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c[:-1])) for c in CASES])
def test_mid_tiles(case):
    import torch
    torch.backends.cuda.matmul.allow_tf32 = False
    mode, bt, h, ht, v, groups, products = case
    g = torch.Generator(device="cuda")
    g.manual_seed(bt + h + v)
    rnd = lambda r, c, std: (torch.randn(r, c, generator=g, device="cuda") * std).to(torch.bfloat16)
    s, w = rnd(bt, h, 1.0), rnd(v, h, h ** -0.5)
    y = torch.randint(0, v, (bt,), generator=g, device="cuda")
    y[3::7] = -100
    y[::9] = v - 1
    th = rnd(bt, ht, 1.0) if ht else None
    tw = rnd(v, ht, ht ** -0.5) if mode == "separate" else None
    tl = rnd(bt, v, 1.0).float() if mode == "precomputed" else None
    kd, w_t = (0.0, 0.0) if mode == "none" else (0.5, 0.0 if mode == "precomputed" else 1.0)
    teacher = (Teacher.Separate(th, tw) if mode == "separate" else
               Teacher.Precomputed(tl) if mode == "precomputed" else Teacher.Tied(th))
    opts = LossOptions(kd_weight=kd, temperature=1.5, label_smoothing=0.1, teacher_ce_weight=w_t,
                       chunk_size=ChunkSize.Fixed(-(-bt // groups)))
    ctx = H.Context(0)
    if groups > 1:
        ctx.set_staging_budget(1)
    got, names = kernels_of(lambda: H.distillation_loss(s, w, y, teacher, opts, ctx=ctx))
    ctx.close()
    took = {"l": "gemm_kk_mid_logits", "w": "gemm_kmt_mid"}
    assert "".join(c for c, k in took.items() if any(k in n for n in names)) == products
    ref = loss_chunked(s, w, y, "tied" if mode == "none" else mode, th, tw, tl, kd=kd, T=1.5,
                       alpha=0.1, w_t=w_t)
    for k in ("loss", "student_ce", "teacher_ce", "kl"):
        check_scalar(k, getattr(got, k), ref[k])
    for k in ("grad_student_hidden", "grad_weight", "grad_teacher_hidden", "grad_teacher_weight"):
        a, b = getattr(got, k), ref[k]
        assert (a is None) == (b is None), k
        if b is not None:
            check_grad_device(k, a, b, "bf16")
