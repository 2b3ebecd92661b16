"""The calls that users of this framework make, as measurable cases.

Kinds of case (``case["kind"]``) and the use each stands for:

* ``prefill``  select key blocks by mean-pooled scores, then the fused forward
               (``select_mean_pooled`` + ``bsattn_forward``): inference of the
               block-sparse models;
* ``train``    the same with the backward through the autograd op (``bsattn``,
               or ``block_sparse_attention`` with a sigmoid output gate);
* ``gqa``      ``blocksparse_forward`` with a Quest selector or, with selector
               ``dense``, every block: one full-attention layer of a GQA hybrid
               model with its output gate, forward only or with the backward;
* ``select``   a selector alone, as a caller that keeps the block list runs it;
* ``mass``     ``block_mass``, the teacher of the oracle selector and of
               self-distillation;
* ``module``   one training step of a ``BlockSparseSSA`` layer.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(1, os.path.abspath("fused-block-sparse-attention_amd"))

import qwen_blocksparse as gqa  # noqa: E402
import ssa_model  # noqa: E402
import triton_kernel as slot_ops  # noqa: E402
from fbsa_amd import ops, selection  # noqa: E402
from fbsa_amd.autograd import block_sparse_attention  # noqa: E402

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # the smallest call: a short fp32 sequence, where launches and latency count
        {"name": "prefill_fp32_4k", "kind": "prefill", "dtype": "fp32", "B": 1, "H": 4, "L": 4096, "D": 64,
         "bs": 64, "topk": 8, "gate": False, "unit": 1.0},
        # a layer of a small language model over 512-token sequences, trained in fp32
        {"name": "module_512", "kind": "module", "dtype": "fp32", "B": 16, "L": 512, "d": 512, "H": 8, "bs": 64,
         "topk": 4, "gate": True, "causal": True},
        # associative-recall training: many short sequences, small blocks, output gate
        {"name": "train_recall_1k", "kind": "train", "dtype": "bf16", "B": 32, "H": 8, "L": 1024, "D": 64,
         "bs": 32, "topk": 4, "gate": True, "out_gate": True, "unit": 1.0},
        # the long-context language-model layer: prefill, and a training step
        {"name": "prefill_262k", "kind": "prefill", "dtype": "bf16", "B": 1, "H": 8, "L": 262144, "D": 64,
         "bs": 64, "topk": 16, "gate": False, "unit": 0.125},
        {"name": "train_262k", "kind": "train", "dtype": "bf16", "B": 1, "H": 8, "L": 262144, "D": 64,
         "bs": 64, "topk": 16, "gate": False, "out_gate": False, "unit": 0.125},
        # a short prompt of no particular length through a GQA layer, fp16
        {"name": "gqa_2k_ragged", "kind": "gqa", "dtype": "fp16", "B": 1, "Hq": 16, "Hkv": 2, "L": 1999, "D": 256,
         "bs": 128, "topk": 4, "selector": "max", "train": False},
        # a long prompt through a GQA layer
        {"name": "gqa_64k", "kind": "gqa", "dtype": "bf16", "B": 1, "Hq": 16, "Hkv": 2, "L": 65536, "D": 256,
         "bs": 128, "topk": 32, "selector": "max", "train": False},
        # fine-tuning a GQA layer on a document of no particular length
        {"name": "gqa_train_16k_ragged", "kind": "gqa", "dtype": "bf16", "B": 1, "Hq": 16, "Hkv": 2, "L": 16301,
         "D": 256, "bs": 128, "topk": 16, "selector": "max", "train": True},
        # the dense path of the same layer: the budget covers every block
        {"name": "gqa_dense_8k", "kind": "gqa", "dtype": "bf16", "B": 1, "Hq": 16, "Hkv": 2, "L": 8192, "D": 256,
         "bs": 128, "topk": 64, "selector": "dense", "train": False},
        # selection at the longest context: 65536 blocks
        {"name": "select_4m", "kind": "select", "dtype": "bf16", "B": 1, "Hq": 8, "Hkv": 8, "L": 4194304, "D": 64,
         "bs": 64, "topk": 16, "selector": "mean"},
        # the two-stage token-max selector on a long prompt
        {"name": "select_two_stage_64k", "kind": "select", "dtype": "bf16", "B": 1, "Hq": 16, "Hkv": 2, "L": 65501,
         "D": 256, "bs": 128, "topk": 32, "selector": "two_stage"},
        # the true block mass of a GQA layer
        {"name": "mass_16k", "kind": "mass", "dtype": "bf16", "B": 1, "Hq": 16, "Hkv": 2, "L": 16384, "D": 256,
         "bs": 128},
    ]


# ------------------------------------------------------------------- drawing
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(("prefill", "train", "gqa", "gqa", "select", "mass", "module"))
    dt = rng.choice(("bf16", "bf16", "fp16", "fp32"))
    if kind in ("prefill", "train"):
        bs = rng.choice((32, 64, 128))
        long = 65536 if dt == "fp32" else 262144
        c = {"kind": kind, "dtype": dt, "B": 1, "H": rng.choice((4, 8)), "L": bs * _log(rng, 8, long // bs),
             "D": rng.choice((32, 64, 64, 128)), "bs": bs, "topk": rng.randint(3, 16), "gate": rng.random() < 0.5,
             "unit": rng.choice((1.0, 0.125))}
        c["B"] = rng.randint(1, max(1, min(32, 32768 // c["L"])))
        if kind == "train":
            c["out_gate"] = rng.random() < 0.3
        return c
    if kind == "module":
        c = {"kind": kind, "dtype": "fp32", "B": 1, "L": _log(rng, 200, 8192), "d": rng.choice((256, 512)),
             "H": rng.choice((4, 8)), "bs": rng.choice((32, 64)), "topk": rng.randint(2, 8),
             "gate": rng.random() < 0.7, "causal": rng.random() < 0.7}
        c["B"] = rng.randint(1, max(1, min(16, 16384 // c["L"])))
        return c
    c = {"kind": kind, "dtype": dt if kind != "mass" else rng.choice(("bf16", "fp16")), "B": rng.choice((1, 1, 2)),
         "Hq": 0, "Hkv": rng.choice((2, 4)), "L": 0, "D": rng.choice((64, 128, 256)), "bs": rng.choice((64, 128))}
    c["Hq"] = c["Hkv"] * rng.choice((1, 4, 8))
    if kind == "mass":
        c["L"] = c["bs"] * _log(rng, 8, 16384 // c["bs"])
    elif kind == "select":
        c["selector"] = rng.choice(("mean", "max", "lasttok", "qmax", "two_stage"))
        if c["selector"] == "mean":
            c["Hkv"] = c["Hq"]
            c["L"] = c["bs"] * _log(rng, 16, 1048576 // c["bs"])
        else:
            c["L"] = _log(rng, 1000, 65536)
        c["topk"] = rng.randint(4, 32)
    else:
        c["selector"] = rng.choice(("max", "max", "dense"))
        c["train"] = rng.random() < 0.5
        c["L"] = _log(rng, 500, 8192 if c["selector"] == "dense" else 32768)
        c["topk"] = rng.randint(4, 32) if c["selector"] == "max" else 1 + c["L"] // c["bs"]
    return c


def _cost(c):
    """Seconds at 60 TFLOP/s in 32 bits, 500 in 16 bits, and 2 TB/s."""
    w = work(c)
    return w["flops"] / (6e13 if c["dtype"] == "fp32" else 5e14) + w["bytes"] / 2e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


# -------------------------------------------------------------------- inputs
def _randn(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def make(*shape, dtype=dt, unit=1.0):
        x = torch.randn(*shape, generator=g, device=DEV, dtype=dtype)
        return x if unit == 1.0 else x.mul_(unit)
    return make


def _selector(case):
    name, topk, bs = case["selector"], case["topk"], case["bs"]
    return {"max": gqa.SelectMax, "lasttok": gqa.SelectLastTok, "qmax": gqa.SelectMaxQMax,
            "two_stage": gqa.SelectTwoStage}[name](topk, bs)


def prepare(case, seed):
    kind, make, st = case["kind"], _randn(case, seed), {"case": case}
    if kind == "module":
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            st["layer"] = ssa_model.BlockSparseSSA(case["d"], case["H"], block=case["bs"], topk=case["topk"],
                                                   gate=case["gate"], causal=case["causal"]).to(DEV)
        st["x"] = make(case["B"], case["L"], case["d"]).requires_grad_(True)
        st["do"] = make(case["B"], case["L"], case["d"])
        return st
    B, L, D = case["B"], case["L"], case["D"]
    if kind in ("prefill", "train"):
        H, unit = case["H"], case["unit"]
        st["q"], st["k"], st["v"] = (make(B, H, L, D, unit=unit) for _ in range(3))
        nblk = L // case["bs"]
        kk = 1 + min(case["topk"], nblk - 1)
        st["gate"] = F.logsigmoid(make(B, nblk, kk, dtype=torch.float32)) if case["gate"] else None
        if kind == "train":
            for n in "qkv":
                st[n].requires_grad_(True)
            st["do"] = make(B, H, L, D)
            st["out_gate"] = make(B, H, L, D).requires_grad_(True) if case["out_gate"] else None
        return st
    Hq, Hkv = case["Hq"], case["Hkv"]
    st["q"], st["k"] = make(B, Hq, L, D), make(B, Hkv, L, D)
    if kind == "gqa":
        # values and the output gate come straight from their projections
        st["v"] = make(B, L, Hkv, D).transpose(1, 2)
        st["out_gate"] = make(B, L, Hq, D).transpose(1, 2)
        if case["train"]:
            for n in ("q", "k", "v", "out_gate"):
                st[n].requires_grad_(True)
            st["do"] = make(B, Hq, L, D)
    if kind in ("gqa", "select") and case["selector"] not in ("dense", "mean"):
        st["selector"] = _selector(case)
    return st


# ---------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "module":
        layer, x = state["layer"], state["x"]
        out = layer(x)
        params = [p for n, p in layer.named_parameters() if layer.gate or not n.startswith("sel_")]
        return [out.detach(), *torch.autograd.grad(out, [x, *params], state["do"])]
    if kind == "mass":
        return gqa.block_mass(state["q"], state["k"], case["bs"])
    if kind == "select":
        if case["selector"] == "mean":
            return selection.select_mean_pooled(state["q"], state["k"], case["bs"], case["topk"], causal=True)
        return state["selector"].select(state["q"], state["k"])
    q, k, v = state["q"], state["k"], state["v"]
    if kind == "gqa":
        if not case["train"]:
            with torch.no_grad():
                return gqa.blocksparse_forward(q, k, v, selector=state.get("selector"), topk=case["topk"],
                                               bs=case["bs"], out_gate=state["out_gate"])
        o = gqa.blocksparse_forward(q, k, v, selector=state.get("selector"), topk=case["topk"], bs=case["bs"],
                                    out_gate=state["out_gate"])
        return [o.detach(), *torch.autograd.grad(o, (q, k, v, state["out_gate"]), state["do"])]
    sel = selection.select_mean_pooled(q, k, case["bs"], case["topk"], causal=True)
    if kind == "prefill":
        return [sel, slot_ops.bsattn_forward(q, k, v, sel, state["gate"], causal=True)]
    if case["out_gate"]:
        gate = state["gate"].unsqueeze(1) if state["gate"] is not None else None
        o = block_sparse_attention(q, k, v, sel.unsqueeze(1), mask=ops.MASK_SLOT_CAUSAL, gate=gate,
                                   out_gate=state["out_gate"])
        return [sel, o.detach(), *torch.autograd.grad(o, (q, k, v, state["out_gate"]), state["do"])]
    o = slot_ops.bsattn(q, k, v, sel, state["gate"], causal=True)
    return [sel, o.detach(), *torch.autograd.grad(o, (q, k, v), state["do"])]


# ---------------------------------------------------------------------- work
def work(case):
    """Inputs read once and outputs written once; multiply-adds of the valid
    (query block, key block) pairs, each gradient product once more."""
    kind, s, B, L = case["kind"], 4 if case["dtype"] == "fp32" else 2, case["B"], case["L"]
    bs = case["bs"]
    nblk = -(-L // bs)
    if kind == "module":
        d, kk = case["d"], 1 + min(case["topk"], nblk - 1)
        pairs = sum(min(i + 1, kk) if case["causal"] else kk for i in range(nblk))
        lin = 2 * B * L * (4 * d * d + 2 * (d * 32 + 32 * 32))
        par = 4 * (4 * d * d + 2 * (d * 32 + 32 * 32))
        return {"bytes": 4 * B * L * d * 4 + 2 * par, "flops": 3 * lin + 3.5 * 4 * B * pairs * bs * bs * d}
    Hq, Hkv, D = case.get("Hq", case.get("H")), case.get("Hkv", case.get("H")), case["D"]
    qb, kb = B * Hq * L * D * s, B * Hkv * L * D * s
    if kind == "mass":
        return {"bytes": qb + kb + 4 * B * Hkv * nblk * nblk, "flops": B * Hq * L * L * D}
    # scored block pairs: pooled vectors, or every token's for the token-max selectors
    name = case.get("selector", "mean")
    groups = 1 if name == "mean" else Hkv
    score = {"mean": 1, "dense": 0, "max": 2, "lasttok": 2, "qmax": 2 * bs, "two_stage": 2}[name]
    pick = B * groups * score * nblk * nblk * D
    if name == "two_stage":
        pick += 4 * B * Hkv * bs * D * sum(min(i + 1, 4 * case["topk"]) for i in range(nblk))
    if kind == "select":
        kk = 1 + min(case["topk"], nblk)
        return {"bytes": (qb // bs if name == "lasttok" else qb) + kb + B * groups * nblk * kk * 4, "flops": pick}
    if name == "dense":
        pairs = nblk * (nblk + 1) // 2
    else:
        extra = 1 if kind != "gqa" else 2
        pairs = sum(min(i + 1, case["topk"] + extra) for i in range(nblk))
    attn = 4 * B * Hq * pairs * bs * bs * D
    if kind == "prefill" or (kind == "gqa" and not case["train"]):
        return {"bytes": (3 if kind == "gqa" else 2) * qb + 2 * kb, "flops": pick + attn}
    gated = 2 if kind == "gqa" or case["out_gate"] else 0
    return {"bytes": (4 + gated) * qb + 4 * kb, "flops": pick + 3.5 * attn}


def tolerance(case):
    """About four times the error against 64 bits that each type was measured at."""
    if case["kind"] == "select":
        return "exact"
    if case["kind"] == "module":  # the selector's bias gradients cancel to 1e-3 of their terms
        return {"rel": 6e-5, "max": 1e-3}
    if case["kind"] == "mass":  # fp32 sums of scores rounded to 16 bits; a few land on the other side
        return {"rel": 2e-5, "max": 2e-3}
    return {"fp32": {"rel": 1e-5, "max": 1e-3}, "fp16": {"rel": 2e-3, "max": 0.05}, "bf16": {"rel": 1e-2, "max": 0.2}}[
        case["dtype"]]


# ------------------------------------------------- the same in 64 bits (torch)
def _rnd(x, dt):
    return x if dt == torch.float32 else x.to(dt).double()


def _blocks(x, bs):
    B, H, L, D = x.shape
    return F.pad(x, (0, 0, 0, -L % bs)).reshape(B, H, -1, bs, D)


def _mean_scores(q, k, bs, dt):
    """Scores of mean-pooled blocks, rounded where the operand type rounds."""
    def pool(x):
        out = [_rnd(_blocks(x[:, h:h + 1].double(), bs).mean(3), dt) for h in range(x.shape[1])]
        return _rnd(torch.stack([o[:, 0] for o in out], 1).mean(1), dt)
    return _rnd(pool(q) @ pool(k).transpose(-1, -2), dt).unsqueeze(1)


def _quest_scores(q, k, bs, dt):
    B, Hq, L, D = q.shape
    Hkv = k.shape[1]
    qg = torch.stack([q[:, h * (Hq // Hkv):(h + 1) * (Hq // Hkv)].double().mean(1) for h in range(Hkv)], 1)
    qp = _rnd(_blocks(_rnd(qg, dt), bs).mean(3), dt)
    kb = _blocks(k.double(), bs)
    up = _rnd(qp.clamp(min=0) @ kb.amax(3).transpose(-1, -2), dt)
    return _rnd(up + _rnd(qp.clamp(max=0) @ kb.amin(3).transpose(-1, -2), dt), dt)


def _top(score, topk, past):
    """The first topk candidates of every row by descending score (ties: lower
    index), and whether each is one that the row may choose."""
    n = score.shape[-1]
    i, j = torch.arange(n, device=DEV).view(n, 1), torch.arange(n, device=DEV)
    score = score.masked_fill(~past(i, j), -math.inf)
    val, idx = score.sort(dim=-1, descending=True, stable=True)
    return idx[..., :topk], torch.isfinite(val[..., :topk])


def _lists(case, q, k):
    """Key blocks of every query block (B, Hsel, nblk, slots) and the slots in use."""
    bs, dt = case["bs"], DTYPES[case["dtype"]]
    nblk = -(-q.shape[2] // bs)
    own = torch.arange(nblk, device=DEV).view(1, 1, nblk, 1)
    if case["kind"] != "gqa":
        idx, ok = _top(_mean_scores(q, k, bs, dt), min(case["topk"], nblk - 1), lambda i, j: j < i)
        own = own.expand(*idx.shape[:3], 1)
        return torch.cat([own, idx], -1), torch.cat([torch.ones_like(own, dtype=torch.bool), ok], -1)
    if case["selector"] == "dense":
        idx = own.view(1, 1, 1, nblk).expand(q.shape[0], 1, nblk, nblk)
        return idx, idx <= own
    idx, ok = _top(_quest_scores(q, k, bs, dt), min(case["topk"], nblk), lambda i, j: j <= i)
    hit = torch.zeros(*idx.shape[:3], nblk, dtype=torch.bool, device=DEV).scatter_(3, idx, ok)
    hit |= torch.eye(nblk, dtype=torch.bool, device=DEV)
    hit[..., 0] = True
    used, idx = hit.sort(dim=-1, descending=True, stable=True)
    n = int(used.sum(-1).max())
    return idx[..., :n], used[..., :n]


def _attend(q, k, v, idx, used, gate, out_gate, do, bs, causal, scale):
    """Gather attention of query blocks in chunks, and its gradients when do is given."""
    B, Hq, L, D = q.shape
    Hkv, nblk, kk = k.shape[1], idx.shape[2], idx.shape[3]
    qb, kb, vb = (_blocks(t, bs) for t in (q, k, v))
    gb = _blocks(out_gate, bs) if out_gate is not None else None
    dob = _blocks(do, bs) if do is not None else None
    o = torch.zeros(B, Hq, nblk, bs, D, dtype=torch.float64, device=DEV)
    grads = None
    if do is not None:
        grads = [torch.zeros_like(o), *(torch.zeros(B, Hkv, nblk, bs, D, dtype=torch.float64, device=DEV)
                                        for _ in range(2)), torch.zeros_like(o) if gb is not None else None]
    step = max(1, (1 << 25) // (bs * kk * bs))
    t = torch.arange(bs, device=DEV)
    for b in range(B):
        for h in range(Hq):
            hk = h // (Hq // Hkv)
            hs = hk if idx.shape[1] > 1 else 0
            for i0 in range(0, nblk, step):
                i = torch.arange(i0, min(nblk, i0 + step), device=DEV)
                j = idx[b, hs, i]                                              # (n, kk)
                qc = qb[b, h, i].double()
                kc, vc = (x[b, hk, j].double().flatten(1, 2) for x in (kb, vb))  # (n, kk*bs, D)
                s = torch.bmm(qc, kc.transpose(1, 2)).mul_(scale)
                key = (j.unsqueeze(-1) * bs + t).flatten(1)
                ok = used[b, hs, i].repeat_interleave(bs, 1).unsqueeze(1) & (key < L).unsqueeze(1)
                if causal:
                    ok = ok & (key.unsqueeze(1) <= (i.unsqueeze(-1) * bs + t).unsqueeze(-1))
                if gate is not None:
                    s += gate[b, i].double().repeat_interleave(bs, 1).unsqueeze(1)
                p = s.masked_fill_(~ok, -math.inf).softmax(-1)
                a = torch.bmm(p, vc)
                sg = torch.sigmoid(gb[b, h, i].double()) if gb is not None else 1.0
                o[b, h, i] = a * sg
                if do is None:
                    continue
                dc = dob[b, h, i].double()
                if gb is not None:
                    grads[3][b, h, i] = dc * a * sg * (1 - sg)
                    dc = dc * sg
                ds = torch.bmm(dc, vc.transpose(1, 2)).sub_((dc * a).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                grads[0][b, h, i] = torch.bmm(ds, kc)
                flat = j.flatten()
                grads[1][b, hk].index_add_(0, flat, torch.bmm(ds.transpose(1, 2), qc).view(-1, bs, D))
                grads[2][b, hk].index_add_(0, flat, torch.bmm(p.transpose(1, 2), dc).view(-1, bs, D))
    out = [o] + [g for g in grads or [] if g is not None]
    return [x.flatten(2, 3)[:, :, :L] for x in out]


def _exact_module(case, st):
    bs, H, L = case["bs"], case["H"], case["L"]
    w = {n: p.detach().double().requires_grad_(True) for n, p in st["layer"].named_parameters()}
    x = st["x"].detach().double().requires_grad_(True)
    lin = lambda t, n: t @ w[n + ".weight"].t() + w[n + ".bias"]  # noqa: E731
    xp = F.pad(x, (0, 0, 0, -L % bs))
    B, Lp, d = xp.shape
    nblk, dh = Lp // bs, d // H
    q, k, v = (t.view(B, nblk, bs, H, dh).permute(0, 3, 1, 2, 4) for t in lin(xp, "qkv").chunk(3, -1))
    feat = lambda n: lin(F.gelu(lin(xp, n + ".0")), n + ".2").view(B, nblk, bs, -1)  # noqa: E731
    sq, kf = feat("sel_q").mean(2), feat("sel_k")
    raw = torch.maximum(sq @ kf.mean(2).transpose(1, 2), sq @ kf.amax(2).transpose(1, 2))
    idx, ok = _top(raw.detach(), min(case["topk"], nblk - 1),
                   (lambda i, j: j < i) if case["causal"] else (lambda i, j: j != i))
    own = torch.arange(nblk, device=DEV).view(1, nblk, 1).expand(B, nblk, 1)
    j = torch.cat([own, idx], -1)
    ok = torch.cat([torch.ones_like(own, dtype=torch.bool), ok], -1)
    kk = j.shape[-1]
    row = torch.arange(B, device=DEV).view(B, 1, 1)
    kc, vc = (t.transpose(1, 2)[row, j].permute(0, 3, 1, 2, 4, 5).flatten(3, 4) for t in (k, v))
    s = q @ kc.transpose(-1, -2) * dh ** -0.5                        # (B, H, nblk, bs, kk*bs)
    if case["gate"]:
        s = s + F.logsigmoid(raw.gather(2, j)).repeat_interleave(bs, 2)[:, None, :, None]
    t = torch.arange(bs, device=DEV)
    live = ok[:, None, :, None, :, None].expand(B, 1, nblk, bs, kk, bs).clone()
    if case["causal"]:
        live[:, :, :, :, 0] = t.view(bs, 1) >= t
    s = s.masked_fill(~live.flatten(4, 5), -math.inf)
    out = (s.softmax(-1) @ vc).permute(0, 2, 3, 1, 4).reshape(B, Lp, d)[:, :L]
    out = lin(out, "o")
    params = [p for n, p in w.items() if case["gate"] or not n.startswith("sel_")]
    return [out.detach(), *torch.autograd.grad(out, [x, *params], st["do"].double())]


def exact(case, seed):
    kind = case["kind"]
    if kind == "select":
        return None  # block indices: compared as they are
    st = prepare(case, seed)
    if kind == "module":
        return _exact_module(case, st)
    with torch.no_grad():
        if kind == "mass":
            return _exact_mass(case, st)
        q, k, v = (st[n].detach() for n in "qkv")
        og, do = st.get("out_gate"), st.get("do")
        idx, used = _lists(case, q, k)
        out = _attend(q, k, v, idx, used, st.get("gate"), og.detach() if og is not None else None, do, case["bs"],
                      True, case["D"] ** -0.5)
        if kind == "gqa":
            return out if case["train"] else out[0]
        return [None, *out]


def _exact_mass(case, st):
    """Scores rounded to the operand type after the product and after the scale
    (as a 16-bit matmul rounds them), the rest in 64 bits."""
    q, k, bs, dt = st["q"], st["k"], case["bs"], DTYPES[case["dtype"]]
    B, Hq, L, D = q.shape
    Hkv, nblk = k.shape[1], L // bs
    mass = torch.zeros(B, Hkv, nblk, nblk, dtype=torch.float64, device=DEV)
    step = max(bs, (1 << 27) // L // bs * bs)
    key = torch.arange(L, device=DEV)
    for b in range(B):
        for h in range(Hq):
            kt = k[b, h * Hkv // Hq].double().t()
            for r in range(0, L, step):
                s = _rnd(_rnd(q[b, h, r:r + step].double() @ kt, dt) * D ** -0.5, dt)
                s.masked_fill_(key > key[r:r + step].unsqueeze(1), -math.inf)
                p = s.softmax(-1).view(-1, bs, nblk, bs).sum(-1).mean(1)
                mass[b, h * Hkv // Hq, r // bs:r // bs + p.shape[0]] += p / (Hq // Hkv)
    return mass
