"""The calls this library is timed on: the fused distillation loss (forward and
backward in one call, every teacher mode, fp32 and bf16), its autograd form,
the chunk-launcher slot over prepared logits and the INT8 round trip of
grad_W, from the smallest batch of a unit test to the benchmark's size.

A case is a plain dict. ``prepare`` makes its inputs on the GPU, ``run`` makes
one call, ``exact`` recomputes the outputs in float64 with plain torch.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("orda-cutile-rs_amd"))

import orda_hip as H  # noqa: E402
from orda_hip.autograd import distillation_loss_autograd  # noqa: E402

IGNORE = -100
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _loss(name, teacher, dtype, bt, h, v, *, ht=0, kd=0.4, T=1.5, alpha=0.0, w_t=None, int8=False,
          autograd=False):
    """A distillation_loss call; w_t None is the teacher's default CE weight
    (1 for Tied, else 0), teacher "none" is student CE alone."""
    tied = teacher == "tied"
    return {"name": name, "op": "loss", "teacher": teacher, "dtype": dtype, "bt": bt, "h": h,
            "ht": ht, "v": v, "kd": kd, "T": T, "alpha": alpha,
            "w_t": w_t if w_t is not None else (1.0 if tied else 0.0), "int8": int8,
            "autograd": autograd}


def _slot(name, dtype, n, v, *, student_only=False):
    return {"name": name, "op": "slot", "dtype": dtype, "n": n, "v": v, "T": 1.5, "alpha": 0.1,
            "student_only": student_only}


def _quant(name, rows, cols, *, stochastic=False):
    return {"name": name, "op": "quant", "rows": rows, "cols": cols, "stochastic": stochastic}


def listed():
    return [
        # the reference's CPU-runnable configuration: a unit-test or CI step,
        # where launches and latency count
        _loss("tied_f32_256x512x8192", "tied", "f32", 256, 512, 8192),
        # the fp32 configurations: one chunk-loop step of a 32k-vocabulary
        # model with each teacher mode
        _loss("tied_f32_2048x4096x32000", "tied", "f32", 2048, 4096, 32000),
        _loss("separate_f32_4096x2048x4096x32000", "separate", "f32", 4096, 2048, 32000, ht=4096,
              kd=0.5, T=2.0, alpha=0.1, w_t=1.0),
        _loss("precomputed_f32_4096x4096x65536", "precomputed", "f32", 4096, 4096, 65536, kd=0.7,
              T=1.0),
        # the benchmark: a full training batch at a 131k vocabulary, INT8 grad_W
        _loss("tied_bf16_8192x4096x131072_int8", "tied", "bf16", 8192, 4096, 131072, alpha=0.1,
              int8=True),
        # the same two-model set-ups in the training dtype
        _loss("separate_bf16_4096x2048x4096x32000", "separate", "bf16", 4096, 2048, 32000, ht=4096,
              kd=0.5, T=2.0, alpha=0.1, w_t=1.0),
        _loss("precomputed_bf16_4096x4096x65536", "precomputed", "bf16", 4096, 4096, 65536, kd=0.7,
              T=1.0),
        # a short micro-batch of a small model through autograd, odd vocabulary
        _loss("autograd_bf16_300x768x50257", "tied", "bf16", 300, 768, 50257, alpha=0.1,
              autograd=True),
        # student cross-entropy alone (no teacher term), ragged batch
        _loss("ce_bf16_777x2048x32000", "none", "bf16", 777, 2048, 32000, kd=0.0, T=1.0),
        # the row kernels over logits the caller has: one chunk of the
        # benchmark's plan, and a ragged bf16 one
        _slot("slot_f32_512x131072", "f32", 512, 131072),
        _slot("slot_bf16_100x50257", "bf16", 100, 50257),
        # INT8 round trip of a finished grad_W on its own
        _quant("quant_32000x4096", 32000, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["loss"] * 7 + ["slot"] * 2 + ["quant"])
    odd = rng.random() < 0.4

    def size(lo, hi, step):
        x = _log_int(rng, lo, hi)
        return x if odd else max(step, x // step * step)

    if op == "slot":
        c = _slot("", rng.choice(["f32", "bf16"]), size(16, 1024, 8), size(2048, 152064, 64),
                  student_only=rng.random() < 0.2)
        c["n"] = min(c["n"], (512 * 131072) // c["v"])
    elif op == "quant":
        c = _quant("", size(2048, 131072, 64), size(256, 8192, 64), stochastic=rng.random() < 0.3)
    else:
        teacher = rng.choice(["tied", "tied", "separate", "precomputed", "none"])
        dtype = rng.choice(["f32", "bf16", "bf16"])
        bt, v = size(64, 8192, 16), size(2048, 152064, 64)
        h, ht = size(256, 8192, 64), size(256, 8192, 64)
        kd = 0.0 if teacher == "none" else rng.choice([0.3, 0.5, 1.0])
        c = _loss("", teacher, dtype, bt, h, v, ht=ht if teacher == "separate" else 0, kd=kd,
                  T=rng.choice([1.0, 1.5, 2.0]), alpha=rng.choice([0.0, 0.1]),
                  w_t=rng.choice([0.0, 1.0]) if teacher in ("tied", "separate") else 0.0,
                  int8=rng.random() < 0.2, autograd=rng.random() < 0.3)
        # never more than the largest listed cases (by time: an fp32 flop
        # takes about ten times a bf16 one)
        most = 5e13 if dtype == "bf16" else 4.5e12
        while _flops(c) > most:
            c["bt"] = c["bt"] // 2 + (1 if odd else 0)
            if c["bt"] < 128:
                c["v"] = c["v"] // 2 + (1 if odd else 0)
    del c["name"]
    return c


def _needs_teacher(c):
    return c["kd"] > 0 or c["w_t"] > 0


def _flops(c):
    """The logits, grad_hidden and grad_W products."""
    bt, h, v, t = c["bt"], c["h"], c["v"], 2 if c["w_t"] > 0 else 0
    mac = 3 * bt * h * v
    if c["teacher"] == "tied" and _needs_teacher(c):
        mac += (1 + t) * bt * h * v
    elif c["teacher"] == "separate" and _needs_teacher(c):
        mac += (1 + t) * bt * c["ht"] * v
    return 2.0 * mac


def work(case):
    c = case
    if c["op"] == "quant":
        n = c["rows"] * c["cols"]
        return {"bytes": 9.0 * n + 4 * c["rows"], "flops": 4.0 * n}
    if c["op"] == "slot":
        n, v, es = c["n"], c["v"], 4 if c["dtype"] == "f32" else 2
        return {"bytes": 2.0 * n * v * es + (2 if c["student_only"] else 3) * n * v * 4.0,
                "flops": 20.0 * n * v}
    es = 4 if c["dtype"] == "f32" else 2
    bt, h, v, ht = c["bt"], c["h"], c["v"], c["ht"]
    gs = es if c["autograd"] else 4    # autograd returns gradients in the input dtype
    b = (es + gs) * (bt * h + v * h) + 8 * bt
    if c["teacher"] == "tied":
        b += bt * h * (es + (gs if c["w_t"] > 0 else 0))
    elif c["teacher"] == "separate":
        b += (bt + v) * ht * (es + (gs if c["w_t"] > 0 else 0))
    elif c["teacher"] == "precomputed":
        b += 4 * bt * v
    return {"bytes": float(b), "flops": _flops(c)}


def _make(c, seed):
    """The tensors of a case: hidden rows of unit scale, weights that give
    logits of a few units, a teacher near its student (Precomputed: a peaked
    one), uniform labels with one row in sixteen ignored."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(rows, cols, std, dtype=torch.float32):
        return torch.empty((rows, cols), device="cuda").normal_(0.0, std, generator=g).to(dtype)

    if c["op"] == "quant":
        m = normal(c["rows"], c["cols"], 1e-5)
        y = torch.randint(0, c["rows"], (min(4096, c["rows"]),), device="cuda", generator=g)
        return {"m": m, "y": y}
    if c["op"] == "slot":
        n, v = c["n"], c["v"]
        lg = normal(2 * n, v, 2.0)
        lg[n:] = 0.6 * lg[n:] + 0.8 * lg[:n]
        y = torch.randint(0, v, (n,), device="cuda", generator=g).to(torch.int32)
        return {"logits": lg.to(DTYPES[c["dtype"]]), "y": y}
    bt, h, v, dt = c["bt"], c["h"], c["v"], DTYPES[c["dtype"]]
    s = normal(bt, h, 1.0)
    d = {"s": s.to(dt), "w": normal(v, h, 1.5 / math.sqrt(h), dt)}
    y = torch.randint(0, v, (bt,), device="cuda", generator=g)
    y[torch.rand((bt,), device="cuda", generator=g) < 1 / 16] = IGNORE
    if c["teacher"] == "tied":
        d["th"] = (0.8 * s + 0.6 * normal(bt, h, 1.0)).to(dt)
    elif c["teacher"] == "separate":
        d["th"] = normal(bt, c["ht"], 1.0, dt)
        d["tw"] = normal(v, c["ht"], 1.5 / math.sqrt(c["ht"]), dt)
    elif c["teacher"] == "precomputed":
        d["tl"] = normal(bt, v, 2.0)
        d["tl"][torch.arange(bt, device="cuda"), y.clamp(min=0)] += 8.0
    elif c["teacher"] == "none":
        d["th"] = s.to(dt)     # Tied with both teacher weights 0: not read
    d["y"] = y
    return d


def prepare(case, seed):
    c = case
    st = {"case": c, **_make(c, seed)}
    if c["op"] != "loss":
        return st
    st["opts"] = H.LossOptions(kd_weight=c["kd"], temperature=c["T"], label_smoothing=c["alpha"],
                               teacher_ce_weight=c["w_t"],
                               config=H.KernelConfig(quantize_grad_weight=c["int8"]))
    if c["autograd"]:
        for k in ("s", "w") + (("th", "tw") if c["w_t"] > 0 else ()):
            if k in st:
                st[k].requires_grad_(True)
    if c["teacher"] == "separate":
        st["teacher"] = H.Teacher.Separate(st["th"], st["tw"])
    elif c["teacher"] == "precomputed":
        st["teacher"] = H.Teacher.Precomputed(st["tl"])
    else:
        st["teacher"] = H.Teacher.Tied(st["th"])
    return st


def run(state):
    c = state["case"]
    if c["op"] == "quant":
        return H.quant_rows_int8(state["m"], state["y"], IGNORE, c["stochastic"], 7)
    if c["op"] == "slot":
        out = H.kl_ce_on_logits_chunk(state["logits"], state["y"], c["n"], 1.0 / c["T"], 0.4 * c["T"],
                                      c["T"] * c["T"], 1.0, 1.0, c["alpha"], IGNORE,
                                      c["student_only"], True)
        return {k: out[k] for k in ("grad_kl_student", "kl_per_row", "grad_ce", "ce_loss")}
    if c["autograd"]:
        leaves = {k: state[k] for k in ("s", "w", "th", "tw")
                  if k in state and state[k].requires_grad}
        loss, parts = distillation_loss_autograd(state["s"], state["w"], state["y"],
                                                 state["teacher"], state["opts"])
        grads = torch.autograd.grad(loss, list(leaves.values()))
        return {"loss": loss, "parts": parts, **{"g" + k: g for k, g in zip(leaves, grads)}}
    o = H.distillation_loss(state["s"], state["w"], state["y"], state["teacher"], state["opts"])
    out = {"loss": o.loss, "student_ce": o.student_ce, "teacher_ce": o.teacher_ce, "kl": o.kl,
           "gs": o.grad_student_hidden, "gw": o.grad_weight}
    if o.grad_teacher_hidden is not None:
        out["gth"] = o.grad_teacher_hidden
    if o.grad_teacher_weight is not None:
        out["gtw"] = o.grad_teacher_weight
    return out


def tolerance(case):
    if case["op"] == "quant":
        return "exact"
    if case["op"] == "slot":
        return {"rel": 1e-5, "max": 4e-4}
    if case["int8"]:
        # a code next to a rounding boundary may move by one step of its row
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-3, "max": 5e-1}
    # measured against exact(): fp32 gradients up to 4.6e-6 (largest element
    # 3.5e-5), bf16 ones 2.4e-3 (8e-2)
    return {"rel": 1e-2, "max": 4e-1} if case["dtype"] == "bf16" else {"rel": 2e-5, "max": 2e-4}


# ---------------------------------------------------------------- float64
def _rows(x, y, T, alpha):
    """nll and CE gradient of float64 logits x with labels y, and the softmax
    at temperature T (log-probabilities)."""
    n, v = x.shape
    lp = torch.log_softmax(x, 1)
    keep = y != IGNORE
    yy = y.clamp(min=0)
    r = torch.arange(n, device=x.device)
    nll = -(1 - alpha) * lp[r, yy] - (alpha / v) * lp.sum(1)
    g = lp.exp_()
    g -= alpha / v
    g[r, yy] -= 1 - alpha
    g *= keep[:, None]
    return nll * keep, g, torch.log_softmax(x / T, 1), keep


def _exact_loss(c, d):
    bt, v, T, kd, w_t, alpha = c["bt"], c["v"], c["T"], c["kd"], c["w_t"], c["alpha"]
    s, w, y = d["s"].double(), d["w"].double(), d["y"]
    ms = 1.0 / max(1, int((y != IGNORE).sum()))
    need_t = _needs_teacher(c)
    th = d["th"].double() if "th" in d and need_t else None
    tw = d["tw"].double() if "tw" in d else w
    gs, gw = torch.empty_like(s), torch.zeros_like(w)
    gth = torch.empty_like(th) if th is not None and w_t > 0 else None
    gtw = torch.zeros_like(tw) if gth is not None and c["teacher"] == "separate" else None
    sums = [0.0, 0.0, 0.0]
    step = max(1, int(2e9) // (8 * v))
    for a in range(0, bt, step):
        b = min(bt, a + step)
        nll, g, ls, keep = _rows(s[a:b] @ w.T, y[a:b], T, alpha)
        sums[0] += float(nll.sum())
        if need_t:
            xt = th[a:b] @ tw.T if th is not None else d["tl"][a:b].double()
            tnll, tg, lt, _ = _rows(xt, y[a:b], T, alpha)
            sums[1] += float(tnll.sum()) if w_t > 0 else 0.0
            if kd > 0:
                pt = lt.exp()
                sums[2] += float(((pt * (lt - ls)).sum(1) * keep).sum()) * T * T
                g += kd * T * (ls.exp() - pt) * keep[:, None]
            if gth is not None:
                tg *= w_t
                gth[a:b] = ms * (tg @ tw)
                (gtw if gtw is not None else gw).addmm_(tg.T, th[a:b], alpha=ms)
        gs[a:b] = ms * (g @ w)
        gw.addmm_(g.T, s[a:b], alpha=ms)
    if c["int8"]:
        scale = gw.abs().amax(1, keepdim=True).clamp(min=1e-12) / 127
        keep = torch.zeros(v, dtype=torch.bool, device=y.device)
        keep[y[y != IGNORE]] = True
        gw = torch.where(keep[:, None], gw, (gw / scale).round_() * scale)
    sce, tce, kl = (x * ms for x in sums)
    loss = sce + w_t * tce + kd * kl
    if c["autograd"]:
        out = {"loss": torch.tensor(loss, dtype=torch.float64),
               "parts": torch.tensor([sce, tce, kl], dtype=torch.float64), "gs": gs, "gw": gw}
    else:
        out = {"loss": loss, "student_ce": sce, "teacher_ce": tce, "kl": kl, "gs": gs, "gw": gw}
    if gth is not None:
        out["gth"] = gth
    if gtw is not None:
        out["gtw"] = gtw
    return out


def exact(case, seed):
    c = case
    d = _make(c, seed)
    if c["op"] == "quant":
        if c["stochastic"]:
            return None
        m = d["m"].double()
        scale = m.abs().amax(1, keepdim=True).clamp(min=1e-12) / 127
        out = (m / scale).round_() * scale
        out[d["y"]] = m[d["y"]]
        return (out, None, scale.reshape(-1))
    if c["op"] == "slot":
        n, T = c["n"], c["T"]
        x, y = d["logits"].double(), d["y"].long()
        nll, g, ls, _ = _rows(x[:n], y, T, c["alpha"])
        tnll, tg, lt, _ = _rows(x[n:], y, T, c["alpha"])
        pt = lt.exp()
        return {"grad_kl_student": 0.4 * T * (ls.exp() - pt),
                "kl_per_row": (pt * (lt - ls)).sum(1) * T * T,
                "grad_ce": g if c["student_only"] else torch.cat([g, tg]),
                "ce_loss": nll if c["student_only"] else torch.cat([nll, tnll])}
    return _exact_loss(c, d)
