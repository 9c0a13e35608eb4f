"""The work a user of llsa_amd has it do, as plain cases: the sparse attention operators llsa_l1, llsa_l2 and llsa_l3,
forward alone (sampling) and forward + backward (training), from the shortest sequence the operators take to the
longest the benchmark names, and the Z-order token permutation at the model's entry and exit.

A case of an operator: {"op": "l1" | "l2" | "l3", "mode": "infer" | "train", "B", "H", "N", "t1", "t2", "t3" (topk per
level, finest first; 0 where the operator has no such level), "rope": 2-D RoPE in the operator, "norm": qk RMS norm in
the operator, "layout": "bhnd" (contiguous (B,H,N,64)) or "bnhd" (transposed views of (B,N,H,64), what a linear layer
leaves)}.  A case of the permutation: {"op": "permute", "mode", "B", "N", "C"}.

The inputs are smooth fields on a Z-ordered pixel grid plus white noise, the structure of image features (a token count
that is no power of four is the beginning of the Z-order of the enclosing grid); dO is N(0,1).
"""
import math

import torch

import llsa_amd
from llsa_amd.utils.rope_table import rope_table
from llsa_amd.utils.zorder import zorder_perm

D = 64


def _attn(name, op, mode, B, H, N, t1, t2=0, t3=0, rope=False, norm=False, layout="bhnd"):
    return {"name": name, "op": op, "mode": mode, "B": B, "H": H, "N": N, "t1": t1, "t2": t2, "t3": t3, "rope": rope,
            "norm": norm, "layout": layout}


def listed():
    return [
        # one attention layer on a 32 x 32 grid (benchmark configuration 1): sampling one image, where launches count
        _attn("l1_infer_1k", "l1", "infer", 1, 6, 1024, 8),
        # the same layer in a training step on one image
        _attn("l1_train_1k", "l1", "train", 1, 6, 1024, 8, rope=True, layout="bnhd"),
        # benchmark configuration 2: 64 x 64, batch 4
        _attn("l1_train_4k", "l1", "train", 4, 6, 4096, 16),
        # a token count that is not a square, odd batch and head counts, views of a linear layer's output
        _attn("l1_train_odd", "l1", "train", 3, 5, 7168, 12, rope=True, layout="bnhd"),
        # the reference's own harness (B=2, H=4, topk 8, forward only) at 256 x 256 for one pooled level ...
        _attn("l1_infer_64k", "l1", "infer", 2, 4, 65536, 8),
        # ... and at 128 x 128 for two
        _attn("l2_infer_16k", "l2", "infer", 2, 4, 16384, 8, 8, rope=True),
        # benchmark configuration 3, the headline: 128 x 128, batch 2
        _attn("l2_train_16k", "l2", "train", 2, 6, 16384, 16, 16, rope=True),
        # one attention layer of the DiT-S training step (benchmark configuration 4): batch 8, qk norm and RoPE in the operator
        _attn("l2_train_layer", "l2", "train", 8, 6, 16384, 16, 16, rope=True, norm=True, layout="bnhd"),
        # the largest selections the operators take, at a token count that is not a square
        _attn("l2_train_wide", "l2", "train", 1, 3, 49152, 64, 32, rope=True),
        # benchmark configuration 5: 512 x 512
        _attn("l2_train_256k", "l2", "train", 1, 6, 262144, 16, 16, rope=True),
        # three pooled levels on the same grid
        _attn("l3_train_256k", "l3", "train", 1, 6, 262144, 16, 16, 16, rope=True),
        # the tokens of a DiT-S batch into Z-order, and their gradient back
        {"name": "permute_train", "op": "permute", "mode": "train", "B": 8, "N": 16384, "C": 384},
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    op = rng.choice(["l1", "l1", "l1", "l2", "l2", "l2", "l2", "l3", "permute"])
    mode = rng.choice(["infer", "train", "train"])
    if op == "permute":
        side = 2 ** rng.randint(3, 8)
        C = 64 * rng.randint(1, 18)
        return {"op": op, "mode": mode, "B": _log_int(rng, 1, max(1, min(16, (1 << 26) // (side * side * C)))), "N": side * side, "C": C}
    t1, t2, t3 = rng.choice([4, 8, 8, 12, 16, 16, 20, 24, 32, 48, 64]), 0, 0
    if op == "l1":
        N = 1024 * _log_int(rng, 1, 64)
    elif op == "l2":
        N, t2 = 16384 * _log_int(rng, 1, 16), rng.choice([4, 8, 8, 12, 16, 16, 24, 32])
    else:
        N, t2, t3 = 262144 * rng.randint(1, 2), rng.choice([4, 8, 16, 24]), rng.choice([4, 8, 16, 24])
    if op != "l1":
        t1 = min(t1, 16 * t2)
    t1 = min(t1, N // 16)
    t2 = min(t2, N // 256)
    B, H = _log_int(rng, 1, 8), rng.randint(1, 12)
    case = {"op": op, "mode": mode, "B": B, "H": H, "N": N, "t1": t1, "t2": t2, "t3": t3, "rope": rng.random() < 0.7,
            "norm": rng.random() < 0.3, "layout": rng.choice(["bhnd", "bnhd"])}
    # no dearer than the listed ones: wide selections and the dense selection of one pooled level (which grows with N^2)
    # cost more per operation than the largest listed case
    flops = 0.55e12 if op == "l1" else 1.25e12
    while work(case)["flops"] > flops or case["B"] * case["H"] * N > 2 ** 21:
        if case["B"] > 1:
            case["B"] -= 1
        else:
            case["H"] -= 1
    return case


def _smooth(gen, B, H, N, dev):
    """(B, H, N, 64) fp32: 0.7 x a periodic Gaussian random field of unit variance (length scale 8 pixels) + 0.3 x white
    noise on the smallest power-of-two grid that holds N tokens, first N tokens of its Z-order."""
    W = 1
    while W * W < N:
        W *= 2
    d = torch.arange(W, device=dev, dtype=torch.float32)
    d = torch.minimum(d, W - d)
    kern = torch.exp(-d * d / 128.0)
    i = torch.arange(W, device=dev)
    circ = kern[(i[:, None] - i[None, :]) % W]                     # the periodic convolution as a matrix
    order = zorder_perm(W)[1][:N].to(dev)
    out = torch.empty(B, H, N, D, device=dev)
    for b in range(B):
        f = torch.randn(H * D, W, W, device=dev, generator=gen)
        f = (f.reshape(-1, W) @ circ).reshape(H * D, W, W).transpose(1, 2).contiguous()
        f = (f.reshape(-1, W) @ circ).reshape(H * D, W * W)
        f = f / f.std(dim=1, keepdim=True)
        f = f[:, order].reshape(H, D, N).transpose(1, 2)
        out[b] = 0.7 * f + 0.3 * torch.randn(H, N, D, device=dev, generator=gen)
    return out


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    train = case["mode"] == "train"
    if case["op"] == "permute":
        side = math.isqrt(case["N"])
        perm, inv = (t.to(torch.int32).to(dev) for t in zorder_perm(side))
        x = torch.randn(case["B"], case["N"], case["C"], device=dev, generator=gen).bfloat16().requires_grad_(train)
        dy = torch.randn(case["B"], case["N"], case["C"], device=dev, generator=gen).bfloat16() if train else None
        return {"case": case, "x": x, "dy": dy, "perm": inv, "inv": perm}
    B, H, N = case["B"], case["H"], case["N"]

    def lay(t):
        t = t.bfloat16()
        return t.transpose(1, 2).contiguous().transpose(1, 2) if case["layout"] == "bnhd" else t

    q, k, v = (lay(_smooth(gen, B, H, N, dev)).requires_grad_(train) for _ in range(3))
    state = {"case": case, "q": q, "k": k, "v": v, "do": None, "rope": None, "norm": None}
    if train:
        state["do"] = lay(torch.randn(B, H, N, D, device=dev, generator=gen))
    if case["rope"]:
        W = 1
        while W * W < N:
            W *= 2
        state["rope"] = rope_table(W, dtype=torch.bfloat16)[:N].contiguous().to(dev)
    if case["norm"]:
        gq, gk = (1.0 + 0.1 * torch.randn(D, device=dev, generator=gen) for _ in range(2))
        state["norm"] = (gq.requires_grad_(train), gk.requires_grad_(train), 1e-5)
    return state


def _forward(s):
    c = s["case"]
    if c["op"] == "permute":
        return llsa_amd.permute_tokens(s["x"], s["perm"], s["inv"])
    kw = {"rope": s["rope"], "qk_norm": s["norm"]}
    if c["op"] == "l1":
        return llsa_amd.llsa_l1(s["q"], s["k"], s["v"], c["t1"], 16, **kw)
    if c["op"] == "l2":
        return llsa_amd.llsa_l2(s["q"], s["k"], s["v"], c["t1"], c["t2"], 16, **kw)
    return llsa_amd.llsa_l3(s["q"], s["k"], s["v"], c["t1"], c["t2"], c["t3"], 16, **kw)


def run(state):
    if state["case"]["mode"] == "infer":
        with torch.no_grad():
            return {"o": _forward(state)}
    o = _forward(state)
    if state["case"]["op"] == "permute":
        wrt, names, do = [state["x"]], ["dx"], state["dy"]
    else:
        wrt, names, do = [state["q"], state["k"], state["v"]], ["dq", "dk", "dv"], state["do"]
        if state["norm"] is not None:
            wrt, names = wrt + list(state["norm"][:2]), names + ["dgamma_q", "dgamma_k"]
    return dict(zip(["o"] + names, (o.detach(),) + torch.autograd.grad(o, wrt, do)))


def work(case):
    train = case["mode"] == "train"
    if case["op"] == "permute":
        one = 2 * case["B"] * case["N"] * case["C"] * 2 + 4 * case["N"]
        return {"bytes": one * (2 if train else 1), "flops": 0}
    B, H, N = case["B"], case["H"], case["N"]
    levels = {"l1": 1, "l2": 2, "l3": 3}[case["op"]]
    # the keys of a query: its fine blocks, the blocks of the pooled levels its groups selected, the whole coarsest level
    n_kv = 16 * (case["t1"] + (case["t2"] if levels > 1 else 0) + (case["t3"] if levels > 2 else 0)) + N // 16 ** levels
    # the scores of the selection: the coarsest level against itself, then every level's rows against their candidates
    sel = (N // 16 ** levels) ** 2
    if levels > 1:
        sel += N // 16 * 16 * case["t2"]
    if levels > 2:
        sel += N // 256 * 16 * case["t3"]
    flops = B * H * D * (4 * N * n_kv * (1 if not train else 3.5) + 2 * sel)
    tensor = B * H * N * D * 2
    # forward: q, k, v in, o out; backward besides: dO in, dq, dk, dv out
    return {"bytes": tensor * (8 if train else 4) + (2 * N * D if case["rope"] else 0), "flops": flops}


def tolerance(case):
    if case["op"] == "permute":
        return "exact"
    return {"rel": 1e-2}
