"""The chunk-launcher slot's kernels at the edges of their blocks, against
float64: vocabularies around the 4-column vectors, the 2048-column gradient
blocks and the 4096-column segments, more segments than a wave has lanes, rows
that start on any element, several bands of rows, and the flag combinations.

Tolerances: fp32 exponentials and sums of the rows (a few 2^-24 of the largest
terms): 1e-5 relative on gradients (Frobenius; the KL gradient's differences
of two probabilities of a few 1e-6 carry the exponents' rounding, 1.2e-6
measured) beside 1e-6 a row (a probability near 1: its exponent, up to 16,
is held to 2^-21 of it), 1e-6 relative on losses beside the fp32 resolution of log-sums of
up to 20 (2e-6), 1e-6 on the KL.
"""
import pytest

import orda_hip as H

pytestmark = pytest.mark.gpu

IGNORE = -100


def reference(lg, y, n, T, kd, w_s, w_t, alpha, student_only, kl):
    import torch
    v = lg.shape[1]
    x, keep = lg.double(), y != IGNORE
    yy, r = y.clamp(min=0).long(), torch.arange(n, device=lg.device)

    def ce(z, w):
        lp = torch.log_softmax(z, 1)
        nll = -(1 - alpha) * lp[r, yy]
        if alpha > 0:
            nll = nll - alpha / v * lp.sum(1)
        g = lp.exp() - alpha / v
        g[r, yy] -= 1 - alpha
        return torch.where(keep, nll, 0.0), torch.where(keep[:, None], g * w, 0.0)
    nll, g = ce(x[:n], w_s)
    out = {"ce_loss": nll, "grad_ce": g}
    if not student_only:
        tn, tg = ce(x[n:], w_t)
        out = {"ce_loss": torch.cat([nll, tn]), "grad_ce": torch.cat([g, tg])}
    ls, lt = torch.log_softmax(x[:n] / T, 1), torch.log_softmax(x[n:] / T, 1)
    pt = lt.exp()
    out["kl_per_row"] = torch.where(keep, (pt * (lt - ls)).sum(1) * T * T, 0.0) * kl
    out["grad_kl_student"] = torch.where(keep[:, None], kd * T * (ls.exp() - pt), 0.0) * kl
    return out


def check(n, v, dtype, pad=0, student_only=False, kl=True, alpha=0.1):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(n * 7 + v)
    full = torch.empty((2 * n, v + pad), device="cuda").normal_(0, 2.0, generator=g)
    full[n:] = 0.6 * full[n:] + 0.8 * full[:n]
    lg = full.to(dtype)[:, pad:]
    y = torch.randint(0, v, (n,), device="cuda", generator=g).to(torch.int32)
    y[::5] = IGNORE
    y[1::7] = v - 1
    T, kd, w_s, w_t = 1.5, 0.4, 0.7, 0.5
    got = H.kl_ce_on_logits_chunk(lg, y, n, 1.0 / T, kd * T, T * T, w_s, w_t, alpha, IGNORE,
                                  student_only, kl)
    ref = reference(lg, y, n, T, kd, w_s, w_t, alpha, student_only, kl)
    for k, want in ref.items():
        a = got[k].double()
        assert a.shape == want.shape, k
        assert bool(torch.isfinite(a).all()), k
        d = (a - want).norm()
        if k.startswith("grad"):
            assert float(d) <= 1e-5 * float(want.norm()) + 1e-6 * n ** 0.5, (k, float(d / want.norm()))
        else:
            floor = 2e-6 if k == "ce_loss" else 1e-6
            assert float((a - want).abs().max()) <= 1e-6 * float(want.abs().max()) + floor, k


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("v", [1, 3, 4, 5, 2047, 2048, 2051, 4095, 4096, 4097, 8195, 64 * 4096 + 3,
                               70 * 4096])
def test_slot_vocabulary_edges(v, dtype):
    import torch
    check(6, v, getattr(torch, dtype))


@pytest.mark.parametrize("student_only,kl", [(True, True), (False, False), (True, False)])
def test_slot_flags(student_only, kl):
    import torch
    for dtype in (torch.float32, torch.bfloat16):
        check(9, 5003, dtype, pad=3, student_only=student_only, kl=kl, alpha=0.0)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_slot_several_bands(dtype):
    """More than 128 MB of logits a band: three bands (fp32) or two (bf16) of
    aligned rows, the last one short."""
    import torch
    check(300, 131072, getattr(torch, dtype))


def test_slot_masked_vocabulary():
    """A segment of -inf logits in both rows and one in the student's alone:
    CE and its gradients as float64 gives them, the KL inf or NaN as its terms
    are (0·inf), the KL gradient p_s - p_t."""
    import torch
    n, v = 4, 3 * 4096
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    lg = torch.empty((2 * n, v), device="cuda").normal_(0, 2.0, generator=g)
    lg[:, 4096:8192] = -float("inf")
    y = torch.full((n,), 9000, device="cuda", dtype=torch.int32)
    got = H.kl_ce_on_logits_chunk(lg, y, n, 1.0, 0.4, 1.0, 1.0, 1.0, 0.0, IGNORE, False, True)
    ref = reference(lg, y, n, 1.0, 0.4, 1.0, 1.0, 0.0, False, 1.0)
    for k in ("grad_ce", "grad_kl_student", "ce_loss"):
        d = (got[k].double() - ref[k]).norm()
        assert float(d) <= 1e-5 * float(ref[k].norm()), k
    assert bool(torch.isnan(got["kl_per_row"]).all())
    lg[n:, 4096:8192] = 0.0
    got = H.kl_ce_on_logits_chunk(lg, y, n, 1.0, 0.4, 1.0, 1.0, 1.0, 0.0, IGNORE, False, True)
    assert bool(torch.isposinf(got["kl_per_row"]).all())


@pytest.mark.parametrize("alpha", [0.0, 0.1])
@pytest.mark.parametrize("v,lo", [(4097, 4096), (8193, 8192), (64 * 4096 + 1, 64 * 4096), (3 * 4096, 4096)])
def test_slot_keeps_nan(v, lo, alpha):
    """A row pair with NaN throughout one segment of either row (a last segment
    of one column, a whole one): the losses and gradients that read that row
    are NaN in every column, the others what they are without it."""
    import torch
    n, hi = 3, min(lo + 4096, v)
    g = torch.Generator(device="cuda")
    g.manual_seed(v)
    lg = torch.empty((2 * n, v), device="cuda").normal_(0, 2.0, generator=g)
    y = torch.full((n,), 9, device="cuda", dtype=torch.int32)
    call = lambda x: H.kl_ce_on_logits_chunk(x, y, n, 1.0, 0.4, 1.0, 1.0, 1.0, alpha, IGNORE, False, True)
    clean = call(lg)
    lg[0, lo:hi] = float("nan")        # pair 0: the student's row
    lg[n + 1, lo:hi] = float("nan")    # pair 1: the teacher's
    got = call(lg)
    lost = {"ce_loss": [0, n + 1], "grad_ce": [0, n + 1], "kl_per_row": [0, 1], "grad_kl_student": [0, 1]}
    for k, rows in lost.items():
        for r in range(got[k].shape[0]):
            if r in rows:
                assert bool(torch.isnan(got[k][r]).all()), (k, r)
            else:
                assert torch.equal(got[k][r], clean[k][r]), (k, r)


@pytest.mark.parametrize("v", [4096, 32768, 131072])
def test_slot_peaked_student_flat_teacher(v):
    """Student rows with one logit far above the rest beside nearly flat
    teacher rows: the student's exponential sum is about 1 next to the
    teacher's of up to V, so that it must not come from their difference."""
    import torch
    n = 4
    g = torch.Generator(device="cuda")
    g.manual_seed(v)
    lg = torch.empty((2 * n, v), device="cuda").normal_(0, 1.0, generator=g)
    lg[n:] *= 0.3
    lg[:n, 7] = 20.0
    y = torch.randint(0, v, (n,), device="cuda", generator=g).to(torch.int32)
    T, kd = 1.5, 0.4
    got = H.kl_ce_on_logits_chunk(lg, y, n, 1.0 / T, kd * T, T * T, 1.0, 1.0, 0.0, IGNORE, False, True)
    ref = reference(lg, y, n, T, kd, 1.0, 1.0, 0.0, False, 1.0)
    d = (got["grad_kl_student"].double() - ref["grad_kl_student"]).norm()
    k, want = got["kl_per_row"].double(), ref["kl_per_row"]
    assert float(d) <= 1e-5 * float(ref["grad_kl_student"].norm())
    assert float((k - want).abs().max()) <= 1e-6 * float(want.abs().max()) + 1e-6
