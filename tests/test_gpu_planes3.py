"""fp32 products over three-plane operands (planes made beforehand from 2^34
operations a call on, by the small products' own kernel below), against a
float64 restatement: widths, vocabularies and row counts that are
not multiples of the 64-element K blocks or the 256-wide tiles, every teacher
mode, gradient rows from the fused and from the chunked row pass, two and more
staging groups, and a memory limit that the planes do not fit. Which form a call
took is read from the kernels it launched.

Tolerance 1e-6 on the gradients (Frobenius norm, relative): a value is held to
2^-27, and each of the six plane products but the first is needed for it. The
smallest ones kept, high times low, are 2^-18 / sqrt(3) = 2.2e-6 of a product
at most and 1.5e-6 in the mean, so that a result without one of them is off by
more than the tolerance; fp32 accumulation over these K leaves 1e-7 to 5e-7.
"""
import numpy as np
import pytest

import torch_reference as R
from helpers import kernels_of, normal, uniform_labels

import orda_hip as H
from orda_hip import ChunkSize, LossOptions, Teacher

pytestmark = pytest.mark.gpu

TOL = 1e-6
GRADS = ("grad_student_hidden", "grad_weight", "grad_teacher_hidden", "grad_teacher_weight")

# name: (mode, bt, h, ht, v, teacher CE weight, staging groups)
CASES = {
    "tied": ("tied", 517, 360, 360, 9001, 1.0, 1),
    "tied-groups": ("tied", 517, 360, 360, 9001, 0.5, 4),
    "tied-no-teacher-ce": ("tied", 640, 448, 448, 8192, 0.0, 1),
    "tied-chunked-rows": ("tied", 1950, 65, 65, 13000, 1.0, 1),
    "separate": ("separate", 430, 72, 520, 13001, 1.0, 1),
    "separate-groups": ("separate", 430, 72, 520, 13001, 1.0, 3),
    "separate-no-teacher-ce": ("separate", 700, 200, 328, 15001, 0.0, 1),
    "precomputed-in-place": ("precomputed", 1150, 264, 0, 11000, 0.0, 1),
    "precomputed-copied": ("precomputed", 1150, 264, 0, 11003, 0.0, 1),
    "student-ce": ("none", 1150, 264, 0, 11003, 0.0, 1),
    # few operations: the small kernel splits the values itself
    "small-tied": ("tied", 90, 100, 100, 3001, 1.0, 1),
    "small-separate": ("separate", 71, 33, 77, 2050, 1.0, 2),
    "small-precomputed": ("precomputed", 129, 130, 0, 1027, 0.0, 1),
    "small-student-ce": ("none", 5, 7, 0, 131, 0.0, 1),
}


def make(name):
    mode, bt, h, ht, v, w_t, groups = CASES[name]
    s, w = normal((bt, h), 1), normal((v, h), 2, 1.0 / np.sqrt(h))
    y = uniform_labels(bt, v, 3)
    y[::9] = -100
    y[1::50] = v - 1
    th = normal((bt, ht), 4) if mode in ("tied", "separate") else None
    tw = normal((v, ht), 5, 1.0 / np.sqrt(ht)) if mode == "separate" else None
    tl = normal((bt, v), 6, 1.5) if mode == "precomputed" else None
    kd = 0.0 if mode == "none" else 0.4
    opts = LossOptions(kd_weight=kd, temperature=1.5, label_smoothing=0.1, teacher_ce_weight=w_t,
                       chunk_size=ChunkSize.Fixed(-(-bt // groups)))
    return mode, s, w, y, th, tw, tl, kd, w_t, opts, groups


def call(torch, made, ctx):
    mode, s, w, y, th, tw, tl, _, _, opts, _ = made
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    if mode == "separate":
        t = Teacher.Separate(dev(th), dev(tw))
    elif mode == "precomputed":
        t = Teacher.Precomputed(dev(tl))
    else:
        t = Teacher.Tied(dev(th if th is not None else s))
    return H.distillation_loss(dev(s), dev(w), dev(y), t, opts, ctx=ctx)


def rel(got, ref):
    got = got.double().cpu().numpy()
    assert np.all(np.isfinite(got))
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("name", sorted(CASES))
def test_planes3_against_float64(name):
    import torch
    made = make(name)
    mode, s, w, y, th, tw, tl, kd, w_t, _, groups = made
    ctx = H.Context(0)
    if groups > 1:
        ctx.set_staging_budget(1)
    ctx.set_timing(True)
    got, names = kernels_of(lambda: call(torch, made, ctx))
    assert ctx.kernel_time("gemm_grad_weight")[1] >= groups
    ctx.close()
    small = name.startswith("small-")
    assert any("bf16x3" in n for n in names) != small
    assert any("small_x3" in n for n in names) == small
    ref = R.loss_f64(s, w, y, mode, th=th, tw=tw, tl=tl, w_t=w_t, kd=kd, T=1.5, alpha=0.1)
    for k in ("loss", "student_ce", "teacher_ce", "kl"):
        assert abs(getattr(got, k) - ref[k]) <= 1e-6 * abs(ref[k]) + 1e-9, k
    for k in GRADS:
        g, r = getattr(got, k), ref[k]
        assert (g is None) == (r is None), k
        if r is not None:
            assert rel(g, r) <= TOL, (k, rel(g, r))


def test_planes3_give_way_to_a_memory_limit():
    """A limit that the plain form fits and the planes (6 bytes an element of
    weights and gradient rows) do not: same plan, results within the fp32
    tolerance, again on a second call, and the workspace stays under it."""
    import torch
    made = make("tied")
    free = H.Context(0)
    want = call(torch, made, free)
    held = free.workspace_bytes()
    free.close()
    _, bt, h, _, v, _, _ = CASES["tied"]
    planes = 6 * (v * h + 2 * bt * v)
    ctx = H.Context(0)
    limit = held - planes // 2
    ctx.set_memory_limit(limit)
    for _ in range(2):
        got, names = kernels_of(lambda: call(torch, made, ctx))
        assert not any("bf16x3" in n for n in names)
        assert ctx.workspace_bytes() <= limit
        assert got.chunk_plan == want.chunk_plan
        for k in GRADS[:3]:
            d = getattr(got, k).double() - getattr(want, k).double()
            assert float(d.norm() / getattr(want, k).double().norm()) <= 1e-5, k
    ctx.close()


# An infinite weight (a vocabulary entry masked out): with hidden rows of one
# sign its logits are -inf, its probabilities 0, and loss and weight gradient
# finite, as an fp32 product gives them; the hidden gradients are 0 times an
# infinity. The smaller call runs on the small kernel. Bounds: fp32 loss terms
# and gradients (1e-4, 1e-3), as against the oracle elsewhere.
@pytest.mark.parametrize("bt,h,v", [(70, 130, 1030), (512, 520, 11008)])
def test_infinite_weight_masks_its_column(bt, h, v):
    import torch
    s, w = np.abs(normal((bt, h), 1)) + np.float32(0.01), normal((v, h), 2, 1.0 / np.sqrt(h))
    y = uniform_labels(bt, v - 2, 3)
    w[v - 2] = -np.inf
    opts = LossOptions(kd_weight=0.0, teacher_ce_weight=0.0, label_smoothing=0.0)
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    got = H.distillation_loss(dev(s), dev(w), dev(y), Teacher.Precomputed(dev(normal((bt, v), 4))), opts)
    x = torch.from_numpy(s).double() @ torch.from_numpy(w).double().T
    p = torch.softmax(x, dim=1)
    yt = torch.from_numpy(y)
    loss = -torch.log_softmax(x, dim=1)[torch.arange(bt), yt].mean().item()
    p[torch.arange(bt), yt] -= 1.0
    gw = (p.T @ torch.from_numpy(s).double() / bt).numpy()
    assert abs(got.student_ce - loss) <= 1e-4 * abs(loss)
    assert rel(got.grad_weight, gw) <= 1e-3
    assert torch.isnan(got.grad_student_hidden).all()


def test_planes3_do_not_depend_on_earlier_calls():
    """Under one memory limit, a call whose planes fit gives the same bits in a
    fresh context and after a call of fewer plane bytes but more memory in
    all, whose planes did not fit."""
    import torch
    v, h = 9000, 360
    w, y = normal((v, h), 2, 1.0 / np.sqrt(h)), uniform_labels(1000, v, 3)
    s, tl = normal((1000, h), 1), normal((1000, v), 6, 1.5)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    opts = LossOptions(kd_weight=0.4, temperature=1.5, teacher_ce_weight=0.0)
    tied = LossOptions(kd_weight=0.4, temperature=1.5, teacher_ce_weight=1.0)
    sd, wd, yd, td = dev(s), dev(w), dev(y), dev(tl)
    large = lambda ctx: H.distillation_loss(sd[:700], wd, yd[:700], Teacher.Tied(dev(s[::-1][:700])), tied, ctx=ctx)
    small = lambda ctx: H.distillation_loss(sd, wd, yd, Teacher.Precomputed(td), opts, ctx=ctx)
    limit = 145_000_000
    fresh, used = H.Context(0), H.Context(0)
    for c in (fresh, used):
        c.set_memory_limit(limit)
    planes = lambda f, c: any("bf16x3" in k for k in kernels_of(lambda: f(c))[1])
    assert planes(small, fresh) and not planes(large, used)
    assert planes(small, used)
    want = small(fresh)
    for _ in range(2):
        got = small(used)
        assert used.workspace_bytes() <= limit
        assert torch.equal(got.grad_weight, want.grad_weight)
        assert torch.equal(got.grad_student_hidden, want.grad_student_hidden)
    fresh.close()
    used.close()


# Row pitches of six bytes an element up to the 32 bits a tile's offsets have
# (256 rows: V or rows of 2.8e6), and past them, where the call keeps to the
# fp32 MFMA. fp32 sums of K terms in order are off by 2^-24 sqrt(K / 2) in the
# mean, 7e-5 for the 2.9e6 of the last case, and other rows by all of it.
@pytest.mark.parametrize("bt,h,v,planes", [(300, 64, 2_700_000, True), (300, 64, 2_900_000, False),
                                           (2_900_000, 256, 64, False)])
def test_planes3_up_to_what_a_tile_reaches(bt, h, v, planes):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(v)
    rand = lambda *n: torch.randn(n, device="cuda", generator=g)
    s, w, y = rand(bt, h), rand(v, h) / h ** 0.5, torch.randint(0, v, (bt,), device="cuda", generator=g)
    opts = LossOptions(kd_weight=0.0, teacher_ce_weight=0.0, label_smoothing=0.0)
    ctx = H.Context(0)
    got, names = kernels_of(lambda: H.distillation_loss(s, w, y, Teacher.Tied(s), opts, ctx=ctx))
    ctx.close()
    assert any("bf16x3" in n for n in names) == planes
    p = torch.softmax(s.double() @ w.double().T, dim=1)
    p[torch.arange(bt, device="cuda"), y] -= 1.0
    p /= bt
    for k, ref in (("grad_student_hidden", lambda: p @ w.double()), ("grad_weight", lambda: p.T @ s.double())):
        r = ref()
        assert float((getattr(got, k).double() - r).norm() / r.norm()) <= 3e-4, k
