"""Measured cases of the packed attention: one layer's attention as the models that call it run it, forward and (where
they train) backward, plus the key / value pass that goes before it.

A case is one call (or one training step's call and its gradients) through a public entry point:

``varlen``    ``varlen.varlen_attn``: a pack of log-normal sequence lengths, causal; ``fused`` adds the layer's query norm,
              partial rotation and output gate.
``sliding``   ``sliding_attention.attend``: causal window; ``images`` adds one bidirectional image span to some sequences.
``hook``      ``hip_attention.attend``: one long causal sequence (a global layer); ``planned`` passes the work list a pack
              builds once for all of its layers, ``fused`` the query norm and rotation.
``global``    ``global_attention.attend``: one sequence per call, differentiable (a global layer in training).
``markers``   ``hip_attention.attend`` with one query per sequence over all of its keys (the last layer of a pack that only
              reads its markers; decode-shaped).
``branched``  ``hip_attention.attend`` over prompts that share a prefix, the keys read through the block plan's row table.
``keys``      ``hip_attention.norm_rope`` on the keys and ``hip_attention.norm`` on the values of one layer.

Ranges that ``draw`` spreads over: 256 to 32,768 packed query rows (16,384 for the differentiable head-size-512 layer,
65,536 keys for the markers layer and the key pass), head sizes 64, 128, 256 and 512 with the head counts of this
repository's workloads, odd and ragged lengths, planned and unplanned, fused and plain, one or many sequences.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

from karpo_decision_amd import global_attention, hip_attention, ops, sliding_attention, varlen, vision, workloads

EPS = 1e-6
#: Elements of one float64 score chunk of the reference (2 GiB).
CHUNK = 1 << 28


def _case(name, kind, **more):
    base = {"name": name, "kind": kind, "tokens": 0, "median": 0, "longest": 0, "heads": 16, "kv_heads": 8,
            "head_dim": 128, "window": -1, "scale": 0.0, "train": False, "fused": False, "planned": False,
            "images": False, "pack": 0}
    base.update(more)
    return base


def listed():
    return [
        # a handful of short prompts: one small launch, where the host path and the planner count
        _case("short-pack", "varlen", tokens=976, median=250, longest=511, heads=8, kv_heads=2, head_dim=64),
        # the full-attention layer of a 0.8B-class model over a serving batch, everything around the product fused
        _case("full-prefill", "varlen", tokens=8192, median=600, longest=4096, fused=True),
        # the same layer in a training step
        _case("full-train", "varlen", tokens=8192, median=600, longest=4096, train=True),
        # a 12B-class sliding-window layer over a batch with images
        _case("sliding-prefill", "sliding", tokens=16384, median=1500, longest=8192, head_dim=256, window=1023,
              images=True),
        # the same layer in a training step, text only
        _case("sliding-train", "sliding", tokens=16384, median=1500, longest=8192, head_dim=256, window=1023,
              train=True),
        # a global layer over one long document, the pack planned once for all layers
        _case("global-prefill", "hook", tokens=32768, heads=32, kv_heads=16, planned=True),
        # a global layer of a training sequence
        _case("global-train", "global", tokens=16384, heads=32, kv_heads=16, train=True),
        # the 31B global layer (head size 512, eight query heads per key head), prefill of one long document
        _case("wide-prefill", "hook", tokens=32768, heads=32, kv_heads=4, head_dim=512),
        # the same layer in training
        _case("wide-train", "global", tokens=16384, heads=32, kv_heads=4, head_dim=512, train=True),
        # the last layer of a 48-sequence pack: one query per sequence over all of its keys
        _case("markers", "markers", tokens=65536, median=900, heads=32, kv_heads=16, sequences=48),
        # four prompts of a shared block and four branches each, keys read through the row table
        _case("branched", "branched", heads=32, kv_heads=16, prompts=4, shared=4096, branches=4, branch=512),
        # keys and values of a 32k-token layer on their way into the attention
        _case("key-pass", "keys", tokens=32768, heads=16, kv_heads=16),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["varlen", "varlen", "sliding", "sliding", "hook", "hook", "global", "global", "markers",
                       "branched", "keys"])
    pack = rng.randrange(1 << 20)
    if kind == "varlen":
        heads, kv_heads, head_dim = rng.choice([(8, 2, 64), (16, 8, 128), (16, 8, 128)])
        train = rng.random() < 0.5
        case = _case("", kind, tokens=size(256, 32768), median=size(100, 2000), longest=4096, heads=heads,
                     kv_heads=kv_heads, head_dim=head_dim, train=train,
                     fused=head_dim == 128 and not train and rng.random() < 0.7)
    elif kind == "sliding":
        train = rng.random() < 0.5
        case = _case("", kind, tokens=size(512, 32768), median=size(300, 3000), longest=8192, head_dim=256,
                     window=rng.choice([511, 1023]), train=train, images=rng.random() < 0.5,
                     scale=0.0 if train else rng.choice([0.0, 1.0]))
    elif kind == "hook":
        heads, kv_heads, head_dim = rng.choice([(32, 16, 128), (32, 4, 512)])
        case = _case("", kind, tokens=size(512, 32768), heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                     planned=rng.random() < 0.5, fused=rng.random() < 0.5)
    elif kind == "global":
        heads, kv_heads, head_dim = rng.choice([(32, 16, 128), (32, 4, 512)])
        case = _case("", kind, tokens=size(512, 32768 if head_dim == 128 else 16384), heads=heads, kv_heads=kv_heads,
                     head_dim=head_dim, train=True)
    elif kind == "markers":
        heads, kv_heads, head_dim = rng.choice([(32, 16, 128), (32, 4, 512)])
        sequences = size(4, 64)
        case = _case("", kind, tokens=size(64 * sequences, 65536), median=900, heads=heads, kv_heads=kv_heads,
                     head_dim=head_dim, sequences=sequences)
    elif kind == "branched":
        case = _case("", kind, heads=32, kv_heads=16, prompts=rng.randint(1, 4), shared=size(256, 4096),
                     branches=rng.randint(2, 4), branch=size(32, 512))
    else:
        heads, head_dim = rng.choice([(16, 128), (8, 256), (4, 512)])
        case = _case("", kind, tokens=size(512, 65536), heads=heads, kv_heads=heads, head_dim=head_dim)
    case["pack"] = pack
    del case["name"]
    return case


# ---- layouts (from the case alone)

def _layout(case):
    """(query bounds, key bounds, key row table or None) of the case's pack."""
    kind = case["kind"]
    if kind == "branched":
        q_cu, k_cu, rows, at = [0], [0], [], 0
        for _ in range(case["prompts"]):
            own = list(range(at, at + case["shared"]))
            at += case["shared"]
            q_cu.append(at)
            rows += own
            k_cu.append(len(rows))
            for _ in range(case["branches"]):
                rows += own + list(range(at, at + case["branch"]))
                at += case["branch"]
                q_cu.append(at)
                k_cu.append(len(rows))
        return q_cu, k_cu, rows
    if kind == "markers":
        rng = np.random.default_rng(case["pack"])
        raw = np.exp(rng.normal(math.log(case["median"]), workloads.SIGMA, size=case["sequences"]))
        lengths = np.maximum(16, np.floor(raw / raw.sum() * case["tokens"])).astype(np.int64)
        at = int(np.argmax(lengths))
        lengths[at] = max(16, lengths[at] + case["tokens"] - int(lengths.sum()))
        return list(range(len(lengths) + 1)), workloads.bounds([int(n) for n in lengths]), None
    if case["median"]:
        cu = workloads.bounds(workloads.lognormal_lengths(case["tokens"], case["median"], 16, case["longest"],
                                                          case["pack"]))
    else:
        cu = [0, case["tokens"]]
    return cu, cu, None


def _spans(case, q_cu):
    """One image of 64 to 280 rows in about a third of the sequences that can hold one."""
    if not case["images"]:
        return []
    rng = np.random.default_rng(case["pack"] + 1)
    spans = []
    for a, b in zip(q_cu[:-1], q_cu[1:]):
        rows = int(rng.integers(64, 281))
        if b - a > rows and rng.random() < 0.34:
            start = a + int(rng.integers(0, b - a - rows + 1))
            spans.append((start, start + rows))
    return spans


def _scale(case):
    return case["scale"] or 1.0 / math.sqrt(case["head_dim"])


def _right(case):
    return -1 if case["kind"] == "markers" else 0


# ---- inputs

def _normal(gen, *shape, rms=False):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if rms:  # what the layer's query and key norms leave
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return x.bfloat16()


def _rope(gen, rows, width):
    angle = torch.rand(rows, width // 2, generator=gen, device="cuda") * 30
    angle = torch.cat((angle, angle), -1)
    return angle.cos().bfloat16(), angle.sin().bfloat16()


def _inputs(case, seed):
    """Seeded tensors of the case, the same for ``prepare`` and ``exact``."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    q_cu, k_cu, rows = _layout(case)
    heads, kv_heads, d = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "keys":
        t = {"k": _normal(gen, case["tokens"], kv_heads, d) * 3, "v": _normal(gen, case["tokens"], kv_heads, d)}
        t["weight"] = (torch.randn(d, generator=gen, device="cuda") * 0.2 + 1).bfloat16()
        t["cos"], t["sin"] = _rope(gen, case["tokens"], d)
        return t
    tq, tk = q_cu[-1], (q_cu[-1] if rows is not None else k_cu[-1])
    t = {"q": _normal(gen, tq, heads, d, rms=not case["fused"]), "k": _normal(gen, tk, kv_heads, d, rms=True),
         "v": _normal(gen, tk, kv_heads, d)}
    if case["fused"]:  # the projection's raw output, and the tables that go with it
        t["q"] = t["q"] * 3
        gated = case["kind"] == "varlen"
        t["weight"] = (torch.randn(d, generator=gen, device="cuda") * 0.2 + (0 if gated else 1)).bfloat16()
        t["cos"], t["sin"] = _rope(gen, tq, d // 4 if gated else d)
        if gated:
            t["gate"] = _normal(gen, tq, heads, d) * 2
    if case["train"]:
        t["grad"] = _normal(gen, tq, heads, d)
    return t


def prepare(case, seed):
    s = SimpleNamespace(case=case, **_inputs(case, seed))
    kind = case["kind"]
    if kind == "keys":
        s.k_norm = SimpleNamespace(weight=s.weight, eps=EPS, with_scale=True)
        s.v_norm = SimpleNamespace(eps=EPS, with_scale=False)
        return s
    q_cu, k_cu, rows = _layout(case)
    s.scale = _scale(case)
    s.max_q = max(b - a for a, b in zip(q_cu[:-1], q_cu[1:]))
    s.max_k = max(b - a for a, b in zip(k_cu[:-1], k_cu[1:]))
    s.q_cu = torch.tensor(q_cu, dtype=torch.int32, device="cuda")
    s.k_cu = torch.tensor(k_cu, dtype=torch.int32, device="cuda")
    s.rows = torch.tensor(rows, dtype=torch.int64, device="cuda") if rows is not None else None
    if s.rows is not None:
        s.rows = ops.key_rows_of(s.rows)
    s.spans = vision.span_tensor(_spans(case, q_cu), "cuda")
    if kind == "global":
        s.lengths = global_attention.lengths(q_cu, k_cu, torch.device("cuda"))
    s.plan = None
    if case["planned"]:
        s.plan = ops.make_plan(q_cu, k_cu, case["heads"], case["kv_heads"], case["head_dim"], -1, 0, device="cuda")
    s.prologue = {}
    if case["fused"]:
        mode = ops.NORM_ONE_PLUS if kind == "varlen" else ops.NORM_WEIGHT
        s.prologue = {"q_norm": ops.Norm(mode, s.weight, EPS), "cos": s.cos, "sin": s.sin}
        if kind == "varlen":
            s.prologue["gate"] = s.gate
    if case["train"]:
        for t in (s.q, s.k, s.v):
            t.requires_grad_()
    return s


# ---- one pass

def _attention(s):
    case, kind = s.case, s.case["kind"]
    if kind == "varlen":
        return varlen.varlen_attn(s.q, s.k, s.v, s.q_cu, s.k_cu, s.max_q, s.max_k, scale=s.scale, window_size=(-1, 0),
                                  enable_gqa=True, **s.prologue)
    if kind == "sliding":
        return sliding_attention.attend(s.q, s.k, s.v, s.q_cu, s.k_cu, s.max_q, s.max_k, s.scale, case["window"],
                                        spans=s.spans)
    if kind == "global":
        return global_attention.attend(s.q, s.k, s.v, s.lengths[0, 0, :1], s.lengths[0, 1, :1], True, s.scale)
    if kind == "markers":
        return hip_attention.attend(s.q, s.k, s.v, s.q_cu, s.k_cu, 1, s.scale)
    return hip_attention.attend(s.q, s.k, s.v, s.q_cu, s.k_cu, s.max_q, s.scale, causal=True, plan=s.plan, rows=s.rows,
                                **s.prologue)


def run(state):
    s = state
    if s.case["train"]:
        out = _attention(s)
        return (out.detach(), *torch.autograd.grad(out, (s.q, s.k, s.v), s.grad))
    with torch.inference_mode():
        if s.case["kind"] == "keys":
            return (hip_attention.norm_rope(s.k_norm, s.k[None], s.cos, s.sin), hip_attention.norm(s.v_norm, s.v[None]))
        return _attention(s)


# ---- what a pass cannot do without

def work(case):
    heads, kv_heads, d = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "keys":
        vectors = 2 * case["tokens"] * kv_heads  # keys and values
        tables = 2 * case["tokens"] * d
        return {"bytes": 2 * (2 * vectors * d + tables), "flops": vectors * d * 6}
    q_cu, k_cu, rows = _layout(case)
    pairs = workloads.allowed_pairs(q_cu, k_cu, case["window"], _right(case), _spans(case, q_cu))
    tq, tk = q_cu[-1], (q_cu[-1] if rows is not None else k_cu[-1])
    q, kv = tq * heads * d, 2 * tk * kv_heads * d
    elements = 2 * q + kv  # q, k, v in, the output out
    products = 2
    if case["fused"]:
        elements += 2 * tq * (d // 4 if case["kind"] == "varlen" else d)
        elements += q if case["kind"] == "varlen" else 0  # the gate
    if case["train"]:
        elements += 2 * q + kv  # the output's gradient in, three gradients out
        products += 5
    return {"bytes": 2 * elements, "flops": 2 * products * d * heads * pairs}


def tolerance(case):
    """bf16 outputs of fp32 sums over bf16 probabilities: 1.7e-3 to 3.1e-3 from the 64-bit result on an MI355X (the
    bf16 rounding of the output alone is 1.7e-3); about four times that."""
    return {"rel": 1e-2}


# ---- the same in 64 bits

def _norm64(x, weight=None):
    x = x.double()
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return x if weight is None else x * weight.double()


def _rope64(x, cos, sin):
    width = cos.shape[-1]
    head, tail = x[..., :width], x[..., width:]
    turned = torch.cat((-head[..., width // 2:], head[..., :width // 2]), -1)
    return torch.cat((head * cos.double()[:, None] + turned * sin.double()[:, None], tail), -1)


def _visible(case, spans, qa, lq, lk, r0, r1, k1):
    """(rows r0..r1 of the sequence, its first k1 keys) bool mask, or None where every key is seen."""
    if _right(case) < 0:
        return None
    i = torch.arange(r0, r1, device="cuda")[:, None] + (lk - lq)
    j = torch.arange(k1, device="cuda")[None, :]
    mask = j <= i
    if case["window"] >= 0:
        mask &= j >= i - case["window"]
    for s0, s1 in spans:
        if s0 >= qa and s1 <= qa + lq:
            x, y = s0 - qa + lk - lq, s1 - qa + lk - lq
            mask |= (i >= x) & (i < y) & (j >= x) & (j < y)
    return mask


def exact(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "keys":
        return _rope64(_norm64(t["k"], t["weight"]), t["cos"], t["sin"])[None], _norm64(t["v"])[None]
    heads, kv_heads, d, train = case["heads"], case["kv_heads"], case["head_dim"], case["train"]
    group, scale = heads // kv_heads, _scale(case)
    q_cu, k_cu, rows = _layout(case)
    spans = _spans(case, q_cu)
    q = t["q"].double()
    if case["fused"]:
        weight = t["weight"].double() + (1 if case["kind"] == "varlen" else 0)
        q = _rope64(_norm64(t["q"]) * weight, t["cos"], t["sin"])
    index = torch.tensor(rows, device="cuda") if rows is not None else None
    out = torch.zeros_like(q)
    if train:
        dq, dk, dv = (torch.zeros(t[n].shape, dtype=torch.float64, device="cuda") for n in ("q", "k", "v"))
    for qa, qb, ka, kb in zip(q_cu[:-1], q_cu[1:], k_cu[:-1], k_cu[1:]):
        lq, lk = qb - qa, kb - ka
        pick = slice(ka, kb) if index is None else index[ka:kb]
        k = t["k"][pick].double().permute(1, 0, 2).contiguous()  # (kv heads, keys, d)
        v = t["v"][pick].double().permute(1, 0, 2).contiguous()
        step = max(1, CHUNK // (heads * lk))
        for r0 in range(0, lq, step):
            r1 = min(lq, r0 + step)
            n = r1 - r0
            reach = lk if _right(case) < 0 else r1 + lk - lq  # keys that any row of the chunk can see
            for s0, s1 in spans:
                if s0 < qa + r1 and s1 > qa + r0:
                    reach = max(reach, s1 - qa + lk - lq)
            first = 0 if case["window"] < 0 or spans else max(0, r0 + lk - lq - case["window"])
            mask = _visible(case, spans, qa, lq, lk, r0, r1, reach)
            ks, vs = k[:, first:reach].contiguous(), v[:, first:reach].contiguous()

            def rows_of(x):  # (n, heads, d) as (kv heads, group * n, d)
                return x[qa + r0:qa + r1].double().view(n, kv_heads, group, d).permute(1, 2, 0, 3).reshape(
                    kv_heads, group * n, d)

            def back(x):
                return x.view(kv_heads, group, n, d).permute(2, 0, 1, 3).reshape(n, heads, d)

            qs = rows_of(q)
            p = torch.matmul(qs, ks.transpose(1, 2).contiguous()).mul_(scale)
            if mask is not None:
                p.view(kv_heads, group, n, -1).masked_fill_(~mask[:, first:], -math.inf)
            p.sub_(p.amax(-1, keepdim=True)).exp_()
            p.div_(p.sum(-1, keepdim=True))
            o = torch.matmul(p, vs)
            out[qa + r0:qa + r1] = back(o)
            if train:
                g = rows_of(t["grad"])
                dv[ka + first:ka + reach] += torch.matmul(p.transpose(1, 2).contiguous(), g).permute(1, 0, 2)
                ds = torch.matmul(g, vs.transpose(1, 2).contiguous())
                ds.sub_((g * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                del p
                dq[qa + r0:qa + r1] = back(torch.matmul(ds, ks))
                dk[ka + first:ka + reach] += torch.matmul(ds.transpose(1, 2).contiguous(), qs).permute(1, 0, 2)
                del ds
    if case["fused"] and case["kind"] == "varlen":
        out *= torch.sigmoid(t["gate"].double())
    return (out, dq, dk, dv) if train else out
