"""The workloads that speed is measured on: First Passage Attention through its public entry points.

`listed()` names the cases, `draw()` gives more of the same ranges, `prepare()` makes what a program holds
before the call and `run()` is one pass.  `exact()` evaluates the same function in float64 with plain torch.

Kinds of case:
  attn   first_passage_attention on (B, H, T, D) tensors, forward alone (no gradient) or with the six
         gradients;
  layer  FirstPassageAttention (projections, Field, attention), forward and backward, fp32 or fp16 autocast;
  field  Field alone, forward and backward;
  lm     FPADecoder's forward to its logits, fp16 autocast, no gradient (evaluation, prompt processing).
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.abspath("first-passage-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import fpa  # noqa: E402
from fpa.lm import FPADecoder  # noqa: E402


def _attn(name, B, H, T, D, dtype, grad, beta="ones", drift=0.0, tau=1.0):
    return dict(name=name, kind="attn", B=B, H=H, T=T, D=D, dtype=dtype, grad=grad, beta=beta, drift=drift, tau=tau)


def listed():
    return [
        # A unit-test or toy-model sized training step in the default dtype: launches and host time.
        _attn("tiny_train_f32", 1, 2, 256, 32, "f32", True),
        # A short prompt of one sequence, ragged length, evaluation only: the smallest latency.
        _attn("short_eval_f16", 1, 12, 200, 64, "f16", False),
        # One sequence of a small model in training: fewer workgroups than the chip holds.
        _attn("one_seq_train_f16", 1, 12, 1000, 64, "f16", True),
        # The headline training shape.
        _attn("train_f16", 4, 12, 2048, 64, "f16", True),
        # Long context, ragged length, drifting phi.
        _attn("long_train_f16", 1, 12, 16381, 64, "f16", True, drift=0.01),
        # Wide heads, long prompt, evaluation only.
        _attn("long_eval_f16_d128", 1, 16, 8192, 128, "f16", False, beta="softplus"),
        # Full-precision training with wide heads, a softplus beta per head.
        _attn("train_f32_d128", 2, 8, 4096, 128, "f32", True, beta="softplus"),
        # Full-precision training at the common head size, ragged length.
        _attn("train_f32_d64", 2, 12, 1500, 64, "f32", True, beta="softplus"),
        # Full-precision evaluation.
        _attn("eval_f32_d64", 4, 12, 2048, 64, "f32", False),
        # The attention layer of the 12-layer language model as it is trained (fp16 autocast).
        dict(name="layer_train_amp", kind="layer", B=8, T=2048, C=768, H=12, amp=True),
        # The layer in full precision at a small model's size.
        dict(name="layer_train_f32", kind="layer", B=4, T=512, C=256, H=4, amp=False),
        # A whole model call: logits of one prompt.
        dict(name="lm_logits_amp", kind="lm", B=1, T=1000, C=768, H=12, layers=4, vocab=32000),
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn"] * 6 + ["layer", "layer", "field"])
    if kind == "attn":
        while True:
            c = dict(kind="attn", B=rng.randint(1, 6), H=rng.choice([1, 2, 4, 6, 8, 12, 16]), T=_loguniform(rng, 64, 16384),
                     D=rng.choice([16, 32, 64, 64, 64, 128, 128]), dtype=rng.choice(["f16", "f16", "f32"]),
                     grad=rng.random() < 0.6, beta=rng.choice(["ones", "softplus"]), drift=rng.choice([0.0, 0.01]),
                     tau=rng.choice([1.0, 1.0, 0.5, 2.0]))
            # no dearer than the largest listed cases
            if work(c)["flops"] * (4 if c["dtype"] == "f32" else 1) <= 9e11 and c["B"] * c["H"] * c["T"] * c["D"] <= 2 ** 25:
                return c
    if kind == "layer":
        H = rng.choice([2, 4, 8, 12])
        D = rng.choice([32, 64, 64])
        return dict(kind="layer", B=rng.randint(1, 8), T=_loguniform(rng, 64, 2048), C=H * D, H=H, amp=rng.random() < 0.5)
    return dict(kind="field", B=rng.randint(1, 8), T=_loguniform(rng, 64, 4096), C=rng.choice([256, 384, 512, 768, 1024]),
                H=rng.choice([4, 8, 12, 16]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "attn":
        B, H, T, D = case["B"], case["H"], case["T"], case["D"]
        dt = torch.float16 if case["dtype"] == "f16" else torch.float32
        q, k, v, do = (_randn(g, B, H, T, D).to(dt) for _ in range(4))
        # phi is a random walk with an optional drift, psi is phi and noise, as Field makes them
        phi = _randn(g, B, H, T).cumsum(-1) - case["drift"] * torch.arange(T, dtype=torch.float32, device="cuda")
        psi = phi + _randn(g, B, H, T)
        beta = torch.ones(H, device="cuda") if case["beta"] == "ones" else F.softplus(_randn(g, H))
        leaves = [q, k, v, phi, psi, beta]
        if case["grad"]:
            leaves = [x.requires_grad_() for x in leaves]
        return dict(case=case, leaves=leaves, do=do)
    with torch.random.fork_rng(devices=["cuda"]):
        torch.manual_seed(seed)
        if case["kind"] == "lm":
            model = FPADecoder(case["vocab"], case["C"], case["H"], case["layers"], 4 * case["C"]).to("cuda")
            tokens = torch.randint(0, case["vocab"], (case["B"], case["T"]), generator=g, device="cuda")
            return dict(case=case, model=model, tokens=tokens)
        if case["kind"] == "layer":
            model = fpa.FirstPassageAttention(case["C"], case["H"]).to("cuda")
        else:
            model = fpa.Field(case["C"], case["H"]).to("cuda")
    x = F.layer_norm(_randn(g, case["B"], case["T"], case["C"]), (case["C"],)).requires_grad_()  # a norm's output
    if case["kind"] == "layer":
        dy = _randn(g, case["B"], case["T"], case["C"])
        return dict(case=case, model=model, x=x, dy=dy.half() if case["amp"] else dy)
    return dict(case=case, model=model, x=x, dphi=_randn(g, case["B"], case["H"], case["T"]),
                dpsi=_randn(g, case["B"], case["H"], case["T"]), dbeta=_randn(g, case["H"]))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["kind"] == "attn":
        leaves = state["leaves"]
        if not case["grad"]:
            with torch.no_grad():
                return fpa.first_passage_attention(*leaves, tau=case["tau"])
        o = fpa.first_passage_attention(*leaves, tau=case["tau"])
        return (o.detach(),) + torch.autograd.grad(o, leaves, state["do"])
    if case["kind"] == "lm":
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            return state["model"](state["tokens"])
    model, x = state["model"], state["x"]
    params = list(model.parameters())
    if case["kind"] == "layer":
        with torch.autocast("cuda", dtype=torch.float16, enabled=case["amp"]):
            y = model(x)
        return (y.detach(),) + torch.autograd.grad(y, [x] + params, state["dy"])
    phi, psi, beta = model(x)
    return (phi.detach(), psi.detach()) + torch.autograd.grad([phi, psi, beta], [x] + params,
                                                              [state["dphi"], state["dpsi"], state["dbeta"]])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    B, T, H = case["B"], case["T"], case["H"]
    pairs = B * H * T * (T + 1) // 2
    if case["kind"] == "attn":
        D, size = case["D"], 2 if case["dtype"] == "f16" else 4
        n, m = B * H * T * D * size, B * H * T * 4
        if not case["grad"]:  # q, k, v, phi, psi read, o written; two products of 2 D per causal pair
            return {"bytes": 4 * n + 2 * m, "flops": 4 * D * pairs}
        # forward, then q, k, v, o, do read and dq, dk, dv, dphi, dpsi written; five more products
        return {"bytes": 4 * n + 2 * m + 8 * n + 4 * m, "flops": 14 * D * pairs}
    C, N = case["C"], B * T
    if case["kind"] == "field":  # x and its gradient, the three projections and their two gradients
        return {"bytes": 4 * (3 * N * C + 4 * N * H), "flops": 3 * 2 * N * C * 3 * H}
    D = C // H
    proj = 2 * N * C * (4 * C + 3 * H)
    if case["kind"] == "layer":
        size = 2 if case["amp"] else 4
        return {"bytes": N * C * (4 + size + size + 4) + 3 * 4 * (4 * C * C), "flops": 3 * proj + 14 * D * pairs}
    L, V = case["layers"], case["vocab"]
    return {"bytes": 4 * (L * 12 * C * C + V * C) + 2 * N * V,
            "flops": L * (proj + 2 * N * 8 * C * C + 4 * D * pairs) + 2 * N * C * V}


def tolerance(case):
    # About four times the largest error against exact() of any output over the listed cases and some eighty
    # drawn ones (rel / max seen: fp32 forward 5e-7 / 7e-6, with gradients 3e-6 / 8e-5; fp16 forward 3e-4 /
    # 3e-3, with gradients 3e-3 / 1.6e-2; layer fp32 1.4e-5 / 3.2e-5, fp16 5.7e-3 / 9e-3; Field 4e-7 / 1.7e-6;
    # logits 2.6e-3 / 5e-2).  dbeta, a sum over all pairs whose terms cancel, sets the figure wherever it is an
    # output; without it the gradients are at 3e-4 (fp16) and 3e-6 (fp32).
    if case["kind"] == "attn":
        if case["dtype"] == "f32":
            return {"rel": 1.5e-5, "max": 3e-4} if case["grad"] else {"rel": 2e-6, "max": 3e-5}
        return {"rel": 1.2e-2, "max": 7e-2} if case["grad"] else {"rel": 1.2e-3, "max": 1.2e-2}
    if case["kind"] == "field":
        return {"rel": 1.6e-6, "max": 7e-6}
    if case["kind"] == "layer":
        return {"rel": 2e-2, "max": 4e-2} if case["amp"] else {"rel": 6e-5, "max": 1.5e-4}
    return {"rel": 1e-2, "max": 0.2}


# ---------------------------------------------------------------------------
# The same in float64, plain torch
# ---------------------------------------------------------------------------

def _rows(q, k, v, phi, psi, beta, tau, t0, t1):
    """Rows t0 .. t1-1 of the attention output from the full tensors, differentiable in all of them."""
    D, n, dev = q.shape[-1], t1 - t0, q.device
    a = -phi / tau
    idx = torch.arange(n, device=dev)
    after = idx[None, :] > idx[:, None]                                      # [s, u]: u after s
    # ranges (s, t] with s and t in the chunk
    own = phi[..., None, t0:t1].expand(*phi.shape[:-1], n, n)
    hard_in = torch.cummin(own.detach().masked_fill(~after, math.inf), -1).values.transpose(-1, -2)
    soft_in = torch.logcumsumexp((-own / tau).masked_fill(~after, -1e30), -1).transpose(-1, -2)
    if t0:
        # ranges that start before the chunk: the part up to t0 - 1 and the part from t0 to t
        head_m = torch.cummin(phi[..., t0:t1].detach(), -1).values[..., :, None]
        head_l = torch.logcumsumexp(a[..., t0:t1], -1)[..., :, None]
        tail = phi[..., 1:t0].detach().flip(-1)
        tail_m = torch.cummin(tail, -1).values.flip(-1) if t0 > 1 else tail
        tail_m = F.pad(tail_m, (0, 1), value=math.inf)[..., None, :]
        tail_l = torch.logcumsumexp(a[..., 1:t0].flip(-1), -1).flip(-1) if t0 > 1 else a[..., 1:t0]
        tail_l = F.pad(tail_l, (0, 1), value=-1e30)[..., None, :]
        hard = torch.cat([torch.minimum(head_m, tail_m), hard_in], -1)
        soft = torch.cat([torch.logaddexp(head_l, tail_l), soft_in], -1)
    else:
        hard, soft = hard_in, soft_in
    past = torch.arange(t1, device=dev)[None, :] < (t0 + idx)[:, None]       # s < t
    soft = (-tau * soft).masked_fill(~past, 0.0)
    hard = hard.masked_fill(~past, math.inf)
    x = (soft - soft.detach()) + torch.where(past, hard, torch.zeros_like(hard)) - psi[..., None, :t1]
    bias = torch.where(past, beta[:, None, None] * x.clamp(max=0.0), torch.zeros_like(x))
    s = torch.matmul(q[..., t0:t1, :], k[..., :t1, :].transpose(-1, -2).contiguous()) / math.sqrt(D) + bias
    causal = torch.arange(t1, device=dev)[None, :] <= (t0 + idx)[:, None]
    return torch.matmul(torch.softmax(s.masked_fill(~causal, -math.inf), -1), v[..., :t1, :])


def _exact_attn(leaves, tau, do=None):
    """o, and with do the six gradients, in float64, chunk of rows by chunk of rows."""
    leaves = [x.detach().double() for x in leaves]
    T, BH = leaves[0].shape[2], leaves[0].shape[0] * leaves[0].shape[1]
    chunk = max(16, min(256, int(2 ** 26 / (BH * T))))
    if do is not None:
        leaves = [x.requires_grad_() for x in leaves]
        grads = [torch.zeros_like(x) for x in leaves]
    o = torch.empty_like(leaves[0], requires_grad=False)
    with torch.set_grad_enabled(do is not None):
        for t0 in range(0, T, chunk):
            t1 = min(T, t0 + chunk)
            rows = _rows(*leaves, tau, t0, t1)
            o[..., t0:t1, :] = rows.detach()
            if do is not None:
                for s, g in zip(grads, torch.autograd.grad(rows, leaves, do[..., t0:t1, :].double())):
                    s += g
    return (o,) + tuple(grads) if do is not None else o


def _field64(x, w, b, H):
    B, T, _ = x.shape
    delta, g, h = F.linear(x, w, b).view(B, T, 3, H).permute(2, 0, 3, 1)
    walk = delta.cumsum(-1)
    return walk + g, walk + h


def _layer64(x, p, H, dy=None):
    """The attention layer on x with the parameters p (name -> float64 tensor); with dy also the gradients."""
    B, T, C = x.shape
    with torch.set_grad_enabled(dy is not None):
        q, k, v = F.linear(x, p["qkv.weight"]).view(B, T, 3, H, C // H).permute(2, 0, 3, 1, 4)
        phi, psi = _field64(x, p["field.proj.weight"], p["field.proj.bias"], H)
        mid = [q, k, v, phi, psi, F.softplus(p["field.beta_raw"])]
    if dy is None:
        o = _exact_attn(mid, 1.0)
        return F.linear(o.transpose(1, 2).reshape(B, T, C), p["out.weight"])
    do = (dy @ p["out.weight"].detach()).view(B, T, H, C // H).transpose(1, 2)
    o, *grads = _exact_attn(mid, 1.0, do)
    flat = o.transpose(1, 2).reshape(B, T, C)
    names = [n for n in p if n != "out.weight"]
    got = torch.autograd.grad(mid, [x] + [p[n] for n in names], grads)
    by = dict(zip(names, got[1:]))
    by["out.weight"] = dy.reshape(-1, C).t().contiguous() @ flat.reshape(-1, C)
    return (F.linear(flat, p["out.weight"].detach()), got[0]) + tuple(by[n] for n in p)


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "attn":
        return _exact_attn(state["leaves"], case["tau"], state["do"] if case["grad"] else None)
    p = {n: w.detach().double() for n, w in state["model"].named_parameters()}
    if case["kind"] == "lm":
        with torch.no_grad():
            norm = lambda y, n: F.layer_norm(y, (case["C"],), p[n + ".weight"], p[n + ".bias"])  # noqa: E731
            x = p["emb.weight"][state["tokens"]]
            for i in range(case["layers"]):
                b = f"blocks.{i}."
                attn = {n[len(b) + 5:]: w for n, w in p.items() if n.startswith(b + "attn.")}
                x = x + _layer64(norm(x, b + "ln1"), attn, case["H"])
                h = F.gelu(F.linear(norm(x, b + "ln2"), p[b + "fc1.weight"], p[b + "fc1.bias"]))
                x = x + F.linear(h, p[b + "fc2.weight"], p[b + "fc2.bias"])
            return F.linear(norm(x, "ln"), p["emb.weight"])
    x = state["x"].detach().double().requires_grad_()
    p = {n: w.requires_grad_() for n, w in p.items()}
    if case["kind"] == "layer":
        return _layer64(x, p, case["H"], state["dy"].double())
    phi, psi = _field64(x, p["proj.weight"], p["proj.bias"], case["H"])
    beta = F.softplus(p["beta_raw"])
    order = [n for n, _ in state["model"].named_parameters()]
    return (phi.detach(), psi.detach()) + torch.autograd.grad(
        [phi, psi, beta], [x] + [p[n] for n in order],
        [state["dphi"].double(), state["dpsi"].double(), state["dbeta"].double()])
