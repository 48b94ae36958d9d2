"""Performance cases of the tree-attention engine.

Each case is one layer-level operation of a tree-training step, called the way
a training program calls it: the tree-masked attention of one decoder layer
(whole trees, partitions over a gateway prefix, scoring without gradients), the
gated-delta-rule layer core of hybrid models, the fused q/k norm + rotary
prologue and the fused leaf loss. ``listed`` holds the named cases, ``draw``
gives further ones of the same ranges.

Shapes: 32 query / 8 key-value heads of 128 (or the 4/2, 16/4 and 16/2 head
layouts of smaller configurations), trees of 47 to 50,109 packed tokens.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from tree_training_amd.attention import tree_attention
from tree_training_amd.conv import tree_conv
from tree_training_amd.gateway import GatewayAccumulator
from tree_training_amd.gdn import GdnTree, gdn_tree, torch_chunk_gated_delta_rule_tree_varlen
from tree_training_amd.hybrid import hybrid_plan
from tree_training_amd.loss import fused_linear_ce
from tree_training_amd.meta import KeyPlan, TreeMetaDevice, build_trees
from tree_training_amd.prologue import qk_prologue
from tree_training_amd.tree import TreeNode
from tree_training_amd.workloads import agent_tree, forest_from_topology, random_forest, rollout_tree, visible_pairs

D = 128
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
# the two-root test forest of the parity tests (47 tokens)
TWO_ROOT = ([3, 4, 3, 4, 5, 3, 3, 4, 4, 3, 4, 3, 4], [-1, 0, 1, 2, 3, 3, 2, 6, -1, 8, 9, 8, 11])


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _attn(name, tree, dtype="bf16", heads=(32, 8), grad=True, plan=True, cut=0):
    return {"name": name, "op": "attn", **tree, "dtype": dtype, "hq": heads[0], "hkv": heads[1], "grad": grad,
            "plan_in_run": plan, "cut": cut}


def _agent(tokens, node_len=(64, 512), depth=6, seed=0):
    return {"tree": "agent", "tokens": tokens, "depth": depth, "lo": node_len[0], "hi": node_len[1],
            "tree_seed": seed}


def _rollout(prompt, leaves, leaf_len=(256, 1024), seed=0):
    return {"tree": "rollout", "prompt": prompt, "leaves": leaves, "lo": leaf_len[0], "hi": leaf_len[1],
            "tree_seed": seed}


def _gdn(name, tree, dtype="bf16", heads=(16, 32), conv=True, truncated=False):
    return {"name": name, "op": "gdn", **tree, "dtype": dtype, "hk": heads[0], "hv": heads[1], "conv": conv,
            "truncated": truncated}


def listed():
    return [
        # the smallest call: the 47-token verification forest in float32, plan
        # and all; launches and latency are what it costs
        _attn("attn_tworoot47_fp32", {"tree": "tworoot"}, dtype="fp32"),
        # a single short rollout group, 1,000-odd tokens in ragged nodes
        _attn("attn_short1k_bf16", _rollout(301, 6, (37, 190), seed=3)),
        # the training step's attention on the 16K agent tree (the headline)
        _attn("attn_agent16k_bf16", _agent(16384)),
        # the same tree cut into 4096-token partitions: every partition attends
        # over its parents' gateway keys, gradients into float32 accumulators
        _attn("attn_gateway16k_bf16", _agent(16384), cut=4096),
        # GRPO-style rollouts: 8K prompt, 64 leaves; the plan is shared by the
        # layers of a model, so it is in hand here
        _attn("attn_rollout48k_bf16", _rollout(8192, 64), plan=False),
        # float32 training runs (gradient verification against per-path runs)
        _attn("attn_agent16k_fp32", _agent(16384), dtype="fp32", plan=False),
        # scoring pass without gradients on a mid-sized ragged tree
        _attn("attn_score5k_bf16", _agent(5003, (33, 391), 5, seed=2), heads=(16, 4), grad=False, plan=False),
        # the hybrid models' linear-attention layer core on the agent tree
        _gdn("gdn_agent16k_bf16", _agent(16384)),
        # its scan alone in float32 on a small ragged forest, through the
        # reference-named function (which also returns the last state)
        _gdn("gdn_scan2k_fp32", _agent(2111, (5, 200), 5, seed=5), dtype="fp32", heads=(4, 8), conv=False),
        # the reference's own truncated arithmetic on whole nodes
        _gdn("gdn_truncated4k_bf16", _agent(4096, seed=1), heads=(8, 16), truncated=True),
        # the attention prologue of a layer, both directions
        {"name": "prologue16k_bf16", "op": "prologue", "tokens": 16318, "hq": 32, "hkv": 8, "dtype": "bf16"},
        # lm_head + cross-entropy of the agent tree's leaf tokens
        {"name": "leafce11k_bf16", "op": "leafce", "rows": 11365, "hidden": 2560, "vocab": 151936, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_tree(rng, lo, hi):
    """A tree of about lo..hi packed tokens (log-uniform), of a drawn kind."""
    n = _log_int(rng, lo, hi)
    kind = rng.choice(["agent", "agent", "rollout", "forest", "chain"])
    seed = rng.randrange(1 << 30)
    if kind == "rollout":
        leaves = rng.randint(2, 64) if n >= 1024 else rng.randint(2, 6)
        prompt = max(1, int(n * rng.uniform(0.1, 0.5)))
        mean = max(2, (n - prompt) // leaves)
        return _rollout(prompt, leaves, (max(1, mean // 2), max(1, mean * 3 // 2)), seed)
    if kind == "forest":
        return {"tree": "forest", "hi": max(2, n // 24), "tree_seed": seed}
    if kind == "chain":
        return {"tree": "chain", "tokens": n, "nodes": rng.randint(1, 9)}
    hi_len = max(4, min(512, n // 6))
    return _agent(n, (max(1, hi_len // 8), hi_len), rng.randint(3, 6), seed)


def draw(rng: random.Random):
    op = rng.choices(["attn", "gateway", "score", "attn32", "gdn", "prologue", "leafce"], [5, 2, 2, 2, 4, 1, 1])[0]
    if op in ("attn", "gateway", "score", "attn32"):
        heads = rng.choice([(32, 8), (32, 8), (16, 4), (4, 2), (16, 2)])
        hi = {"attn": 20000, "gateway": 16384, "score": 20000, "attn32": 6000}[op]
        tree = _draw_tree(rng, 47, hi)
        if op == "gateway":
            tree = _agent(_log_int(rng, 1500, hi), (64, 512), rng.randint(4, 6), rng.randrange(1 << 30))
        cut = _log_int(rng, 600, 4096) if op == "gateway" else 0
        c = _attn("", tree, "fp32" if op == "attn32" else "bf16", heads, op != "score", bool(cut) or
                  rng.random() < 0.5, cut)
    elif op == "gdn":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        heads = rng.choice([(16, 32), (8, 16), (4, 8), (2, 4)])
        trunc = rng.random() < 0.25
        c = _gdn("", _draw_tree(rng, 47, 6000 if trunc else 16384), dtype, heads, rng.random() < 0.6, trunc)
        if trunc and c["tree"] == "chain":      # whole nodes are quadratic: keep them at trajectory length
            c.update({"nodes": max(c["nodes"], c["tokens"] // 512 + 1)})
        if trunc and c["tree"] == "rollout":
            c["prompt"] = min(c["prompt"], 1024)
    elif op == "prologue":
        hq, hkv = rng.choice([(32, 8), (16, 4), (4, 2)])
        c = {"op": "prologue", "tokens": _log_int(rng, 47, 50109), "hq": hq, "hkv": hkv,
             "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    else:
        c = {"op": "leafce", "rows": _log_int(rng, 40, 11365), "hidden": rng.choice([512, 2560]),
             "vocab": rng.choice([1000, 32003, 151936]), "dtype": "bf16"}
    c.pop("name", None)
    return c


def _topology(case):
    kind = case["tree"]
    if kind == "tworoot":
        return TWO_ROOT
    if kind == "agent":
        return agent_tree(case["tree_seed"], case["depth"], (2, 4), (case["lo"], case["hi"]), case["tokens"])
    if kind == "rollout":
        return rollout_tree(case["tree_seed"], case["prompt"], case["leaves"], (case["lo"], case["hi"]))
    if kind == "forest":
        lens, par = random_forest(case["tree_seed"], (1, 2), 4, 3, (1, case["hi"]))
        return lens, par
    n, m = case["tokens"], min(case["nodes"], case["tokens"])
    cuts = [n * i // m for i in range(m + 1)]
    return [b - a for a, b in zip(cuts, cuts[1:])], list(range(-1, m - 1))


def _partitions(topo, cut):
    """The tree's partitions under the token budget, with their gateway bias."""
    roots, _ = forest_from_topology(topo, TreeNode)
    return hybrid_plan(roots, cut)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _rand(gen, *shape, dtype):
    return torch.randn(*shape, device=gen.device, generator=gen, dtype=torch.float32).to(dtype)


def _attn_segments(case, seed):
    """Per problem (the whole tree, or each partition): topology, gateway bias
    and the tensors, token-major as projections leave them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, hq, hkv = DTYPES[case["dtype"]], case["hq"], case["hkv"]
    topo = _topology(case)
    if case["cut"]:
        parts = [(p["node_len"], p["parent"], p["pos_offset"], p.get("bias"), p["past_len"])
                 for p in _partitions(topo, case["cut"])]
    else:
        parts = [(topo[0], topo[1], 0, None, 0)]
    segs = []
    for lens, par, off, bias, lp in parts:
        n = sum(lens)
        s = {"lens": list(lens), "par": list(par), "off": off, "lp": lp, "bias": bias if lp else None,
             "q": _rand(gen, 1, n, hq, D, dtype=dt), "k": _rand(gen, 1, n, hkv, D, dtype=dt),
             "v": _rand(gen, 1, n, hkv, D, dtype=dt), "kp": None, "vp": None}
        if lp:
            s["kp"], s["vp"] = _rand(gen, 1, hkv, lp, D, dtype=dt), _rand(gen, 1, hkv, lp, D, dtype=dt)
        if case["grad"]:
            s["do"] = _rand(gen, 1, n, hq, D, dtype=dt)
        segs.append(s)
    return segs


def _gates(gen, T, hv):
    a = torch.randn(T, hv, device=gen.device, generator=gen)
    b = torch.randn(T, hv, device=gen.device, generator=gen)
    A = torch.rand(hv, device=gen.device, generator=gen) * 16.0 + 1e-3
    return -A * F.softplus(a + 1.0), b.sigmoid()


def _gdn_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lens, par = _topology(case)
    T, hk, hv, dt = sum(lens), case["hk"], case["hv"], DTYPES[case["dtype"]]
    s = {"lens": lens, "par": par}
    if case["conv"]:
        C = 2 * hk * D + hv * D
        s["x"] = _rand(gen, T, C, dtype=dt)
        s["w"] = (0.5 * torch.randn(C, 1, 4, device="cuda", generator=gen)).to(dt)
    else:
        s["q"], s["k"] = _rand(gen, 1, T, hk, D, dtype=dt), _rand(gen, 1, T, hk, D, dtype=dt)
        s["v"] = _rand(gen, 1, T, hv, D, dtype=dt)
    s["g"], s["beta"] = _gates(gen, T, hv)
    s["do"] = _rand(gen, T, hv, D, dtype=dt)
    return s


def _prologue_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, hq, hkv, dt = case["tokens"], case["hq"], case["hkv"], DTYPES[case["dtype"]]
    s = {"q": _rand(gen, T, hq, D, dtype=dt), "k": _rand(gen, T, hkv, D, dtype=dt),
         "qw": (torch.rand(D, device="cuda", generator=gen) + 0.5).to(dt),
         "kw": (torch.rand(D, device="cuda", generator=gen) + 0.5).to(dt),
         "dq": _rand(gen, T, hq, D, dtype=dt), "dk": _rand(gen, T, hkv, D, dtype=dt)}
    pos = torch.randint(0, 4096, (T,), device="cuda", generator=gen)          # depth positions
    inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))
    emb = torch.cat([pos[:, None].float() * inv[None]] * 2, dim=-1)
    s["cos"], s["sin"] = emb.cos().to(dt), emb.sin().to(dt)
    return s


def _leafce_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    N, H, V, dt = case["rows"], case["hidden"], case["vocab"], DTYPES[case["dtype"]]
    labels = torch.randint(0, V, (N,), device="cuda", generator=gen)
    labels[torch.rand(N, device="cuda", generator=gen) < 0.1] = -100          # masked tokens of the leaves
    return {"hidden": _rand(gen, N, H, dtype=dt),
            "weight": (0.02 * torch.randn(V, H, device="cuda", generator=gen)).to(dt), "labels": labels,
            "scale": torch.full((N,), 1.0 / N, device="cuda")}


_INPUTS = {"attn": _attn_segments, "gdn": _gdn_inputs, "prologue": _prologue_inputs, "leafce": _leafce_inputs}


def prepare(case, seed):
    data = _INPUTS[case["op"]](case, seed)
    state = {"case": case, "data": data}
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["op"] == "attn":
        for s in data:
            # transformers' [1, H, T, D] views of the token-major projections
            s["hf"] = [s[n].transpose(1, 2).requires_grad_(case["grad"]) for n in ("q", "k", "v")]
            s["bias"] = s["bias"].to(dev) if s["bias"] is not None else None
        if not case["plan_in_run"]:
            for s in data:
                meta = TreeMetaDevice(s["lens"], s["par"], pos_offset=s["off"], device=dev)
                s["plan"] = KeyPlan(meta.horizon, s["bias"], topo=(s["lens"], s["par"]))
    elif case["op"] == "gdn":
        if case["conv"]:
            state["tree"] = GdnTree(data["lens"], data["par"], dev)
            data["x"].requires_grad_(True)
            data["w"].requires_grad_(True)
        else:
            ends = [0]
            for n in data["lens"]:
                ends.append(ends[-1] + n)
            state["bounds"] = list(zip(ends, ends[1:]))
            for n in ("q", "k", "v"):
                data[n].requires_grad_(True)
        data["g"].requires_grad_(True)
        data["beta"].requires_grad_(True)
    elif case["op"] == "prologue":
        for n in ("q", "k", "qw", "kw"):
            data[n].requires_grad_(True)
    else:
        data["hidden"].requires_grad_(True)
        data["weight"].requires_grad_(True)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_attn(state):
    case, segs = state["case"], state["data"]
    dev = segs[0]["q"].device
    scale = D ** -0.5
    if case["cut"]:                      # a hybrid step builds all partitions' plans at once
        plans = [p for _, p in build_trees([(s["lens"], s["par"], s["off"], s["bias"]) for s in segs], dev)]
    elif case["plan_in_run"]:
        meta = TreeMetaDevice(segs[0]["lens"], segs[0]["par"], device=dev)
        plans = [KeyPlan(meta.horizon, topo=(segs[0]["lens"], segs[0]["par"]))]
    else:
        plans = [s["plan"] for s in segs]
    out = []
    for s, plan in zip(segs, plans):
        q, k, v = s["hf"]
        if not case["grad"]:
            with torch.no_grad():
                out.append(tree_attention(q, k, v, plan, scale))
            continue
        acc = GatewayAccumulator(s["kp"]) if s["lp"] else None
        o = tree_attention(q, k, v, plan, scale, s["kp"], s["vp"], acc)
        out += [o.detach(), *torch.autograd.grad(o, (q, k, v), s["do"])]
        if acc is not None:
            out += [acc.k, acc.v]
    return out


def _run_gdn(state):
    case, s = state["case"], state["data"]
    hk, hv = case["hk"], case["hv"]
    if case["conv"]:
        T = s["x"].shape[0]
        q, k, v = tree_conv(s["x"], s["w"], None, state["tree"], split_sizes=(hk * D, hk * D, hv * D))
        o, _ = gdn_tree(q.view(T, hk, D), k.view(T, hk, D), v.view(T, hv, D), s["g"], s["beta"], state["tree"], None,
                        True, case["truncated"])
        return [o.detach(), *torch.autograd.grad(o, (s["x"], s["w"], s["g"], s["beta"]), s["do"])]
    o, last = torch_chunk_gated_delta_rule_tree_varlen(
        s["q"], s["k"], s["v"], s["g"][None], s["beta"][None], state["bounds"], s["par"], output_final_state=True,
        use_qk_l2norm_in_kernel=True, reference_truncated=case["truncated"])
    return [o.detach(), last.detach(),
            *torch.autograd.grad(o, (s["q"], s["k"], s["v"], s["g"], s["beta"]), s["do"][None])]


def _run_prologue(state):
    s = state["data"]
    qo, ko = qk_prologue(s["q"], s["k"], s["qw"], s["kw"], 1e-6, 1e-6, s["cos"], s["sin"])
    return [qo.detach(), ko.detach(),
            *torch.autograd.grad((qo, ko), (s["q"], s["k"], s["qw"], s["kw"]), (s["dq"], s["dk"]))]


def _run_leafce(state):
    s = state["data"]
    loss = fused_linear_ce(s["hidden"], s["weight"], s["labels"], s["scale"])
    return [loss.detach(), *torch.autograd.grad(loss, (s["hidden"], s["weight"]))]


_RUN = {"attn": _run_attn, "gdn": _run_gdn, "prologue": _run_prologue, "leafce": _run_leafce}


def run(state):
    return _RUN[state["case"]["op"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    e = 2 if case["dtype"] == "bf16" else 4
    if case["op"] == "attn":
        topo = _topology(case)
        T, hq, hkv = sum(topo[0]), case["hq"], case["hkv"]
        P = visible_pairs(topo)          # cutting a tree changes neither the pairs nor the own rows
        past = sum(p["past_len"] for p in _partitions(topo, case["cut"])) if case["cut"] else 0
        fwd = 2 * T * (hq + hkv) + 2 * past * hkv
        if not case["grad"]:
            return {"bytes": e * D * fwd, "flops": 4 * D * hq * P}
        return {"bytes": e * D * (fwd + 2 * T * (hq + hkv)) + 8 * past * hkv * D, "flops": 12 * D * hq * P}
    if case["op"] == "gdn":
        lens, _ = _topology(case)
        T, hk, hv = sum(lens), case["hk"], case["hv"]
        C = (2 * hk + hv) * D
        # in and out: the rows and their gradients, o and do, gates and their gradients
        nbytes = e * T * (2 * C + 2 * hv * D) + 16 * T * hv
        return {"bytes": nbytes, "flops": 18 * D * D * T * hv}
    if case["op"] == "prologue":
        T, H = case["tokens"], case["hq"] + case["hkv"]
        return {"bytes": e * T * D * (4 * H + 2), "flops": 30 * T * H * D}
    N, H, V = case["rows"], case["hidden"], case["vocab"]
    return {"bytes": e * (2 * N * H + 2 * V * H), "flops": 6 * N * H * V}


# About four times the relative errors measured against ``exact``: float32
# 0.2-1.8e-6 (attention's dk, dv the largest), bf16 attention 2.5e-3, bf16
# gated delta rule 3.5e-3 (the conv output is rounded too), bf16 prologue
# 1.7e-3, bf16 leaf loss 3.1e-3 (logits in bf16).
def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": {"attn": 1e-2, "gdn": 1.5e-2, "prologue": 7e-3, "leafce": 1.2e-2}[case["op"]]}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _node_ranges(lens, par):
    """Per node: its token range and those of its ancestors, root first."""
    start, s = [], 0
    for n in lens:
        start.append(s)
        s += n
    paths = []
    for i, p in enumerate(par):
        paths.append((paths[p] if p >= 0 else []) + [(start[i], start[i] + lens[i])])
    return paths


def _exact_attn(case, seed):
    out = []
    for s in _attn_segments(case, seed):
        rep = case["hq"] // case["hkv"]
        heads = lambda t: t[0].double().transpose(0, 1).contiguous()
        q, k, v = heads(s["q"]), heads(s["k"]), heads(s["v"])
        lp = s["lp"]
        if lp:
            k = torch.cat([s["kp"][0].double(), k], dim=1)
            v = torch.cat([s["vp"][0].double(), v], dim=1)
            seen = torch.nonzero(s["bias"].to(q.device) == 0).flatten()
        n, hq, hkv = q.shape[1], q.shape[0], k.shape[0]
        o = torch.zeros_like(q)
        if case["grad"]:
            do = heads(s["do"])
            dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for path in _node_ranges(s["lens"], s["par"]):
            a, b = path[-1]
            for c in range(a, b, 1024):              # query blocks bound the score matrix
                d = min(c + 1024, b)
                own = torch.cat([torch.arange(x, min(y, d), device=q.device) for x, y in path])
                idx = torch.cat([seen, own + lp]) if lp else own
                hide = own[None] > torch.arange(c, d, device=q.device)[:, None]
                if lp:
                    hide = F.pad(hide, (len(seen), 0))
                for g in range(hkv):
                    qq = q[g * rep:(g + 1) * rep, c:d].reshape(-1, D)
                    kk, vv = k[g, idx], v[g, idx]
                    sc = (qq @ kk.t().contiguous()) * D ** -0.5
                    sc.view(rep, d - c, -1).masked_fill_(hide, -math.inf)
                    p = torch.softmax(sc, dim=-1)
                    oo = p @ vv
                    o[g * rep:(g + 1) * rep, c:d] = oo.view(rep, d - c, D)
                    if case["grad"]:
                        dd = do[g * rep:(g + 1) * rep, c:d].reshape(-1, D)
                        ds = p * (dd @ vv.t().contiguous() - (dd * oo).sum(-1, keepdim=True)) * D ** -0.5
                        dq[g * rep:(g + 1) * rep, c:d] = (ds @ kk).view(rep, d - c, D)
                        dk[g].index_add_(0, idx, ds.t().contiguous() @ qq)
                        dv[g].index_add_(0, idx, p.t().contiguous() @ dd)
        out.append(o.transpose(0, 1)[None])
        if case["grad"]:
            out += [dq[None], dk[None, :, lp:], dv[None, :, lp:]]
            if lp:
                out += [dk[:, :lp].transpose(0, 1), dv[:, :lp].transpose(0, 1)]
    return out


def _gdn64(q, k, v, g, beta, lens, par, truncated):
    """Gated delta rule over the tree, 64 bits: per 64-token chunk (or, for
    the truncated rule, per whole node) the within-chunk correction, then the
    state. Returns o [T, Hv, D] and the last node's state."""
    hv, hk = v.shape[1], q.shape[1]
    norm = lambda t: t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    q = (norm(q) * D ** -0.5).repeat_interleave(hv // hk, dim=1)
    k = norm(k).repeat_interleave(hv // hk, dim=1)
    outs, states, start = [], [], 0
    for n, p in zip(lens, par):
        S = states[p] if p >= 0 else torch.zeros(hv, D, D, dtype=q.dtype, device=q.device)
        step = n if truncated else 64
        for c in range(start, start + n, step):
            e = min(c + step, start + n)
            qc, kc, vc = (t[c:e].transpose(0, 1) for t in (q, k, v))
            G = g[c:e].t().cumsum(-1)
            b = beta[c:e].t()[..., None]
            eye = torch.eye(e - c, dtype=q.dtype, device=q.device)
            low = torch.ones_like(eye).tril()
            decay = ((G[:, :, None] - G[:, None, :]) * low).exp() * low
            kt = kc.transpose(1, 2).contiguous()
            R = -(b * (kc @ kt) * decay).tril(-1)
            rhs = torch.cat([b * vc, b * G.exp()[..., None] * kc], dim=-1)
            if truncated:
                X = R @ rhs
                X = rhs + X + R @ X
            else:
                X = torch.linalg.solve_triangular(eye - R, rhs, upper=False, unitriangular=True)
            V = X[..., :D] - X[..., D:] @ S
            outs.append((G.exp()[..., None] * (qc @ S) + ((qc @ kt) * decay) @ V).transpose(0, 1))
            S = G[:, -1:, None].exp() * S + ((G[:, -1:] - G).exp()[..., None] * kc).transpose(1, 2).contiguous() @ V
        states.append(S)
        start += n
    return torch.cat(outs), states[-1]


def _exact_gdn(case, seed):
    s = _gdn_inputs(case, seed)
    lens, par, hk = s["lens"], s["par"], case["hk"]
    T = sum(lens)
    leaf = lambda t: t.detach().double().requires_grad_(True)
    g, beta, do = leaf(s["g"]), leaf(s["beta"]), s["do"].double()
    if case["conv"]:
        x, w = leaf(s["x"]), leaf(s["w"])
        prev = torch.arange(-1, T - 1)
        start = [0]
        for n in lens:
            start.append(start[-1] + n)
        for i, p in enumerate(par):
            prev[start[i]] = start[p + 1] - 1 if p >= 0 else -1
        prev = torch.cat([prev, torch.tensor([-1])])      # index -1: before a root, a zero row
        xz = F.pad(x, (0, 0, 0, 1))
        at, y = torch.arange(T), 0
        for i in range(3, -1, -1):
            y = y + xz[at.to(x.device)] * w[:, 0, i]
            at = prev[at]
        y = F.silu(y)
        q, k, v = (t.view(T, -1, D) for t in torch.split(y, (hk * D, hk * D, case["hv"] * D), dim=1))
        ins = (x, w, g, beta)
    else:
        qkv = [leaf(s[n]) for n in ("q", "k", "v")]
        q, k, v = (t[0] for t in qkv)
        ins = (*qkv, g, beta)
    o, last = _gdn64(q, k, v, g, beta, lens, par, case["truncated"])
    grads = torch.autograd.grad(o, ins, do)
    return [o.detach(), *grads] if case["conv"] else [o.detach()[None], last.detach()[None], *grads]


def _exact_prologue(case, seed):
    s = _prologue_inputs(case, seed)
    ins = [s[n].double().requires_grad_(True) for n in ("q", "k", "qw", "kw")]
    cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
    outs = []
    for x, w in ((ins[0], ins[2]), (ins[1], ins[3])):
        y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w
        a, b = y[..., :D // 2], y[..., D // 2:]
        outs.append(y * cos + torch.cat([-b, a], dim=-1) * sin)
    grads = torch.autograd.grad(outs, ins, (s["dq"].double(), s["dk"].double()))
    return [outs[0].detach(), outs[1].detach(), *grads]


def _exact_leafce(case, seed):
    s = _leafce_inputs(case, seed)
    w = s["weight"].double()
    gh, gw = torch.empty_like(s["hidden"], dtype=torch.float64), torch.zeros_like(w)
    loss = torch.zeros((), dtype=torch.float64, device=w.device)
    wt = w.t().contiguous()
    for c in range(0, case["rows"], 2048):
        h, lab = s["hidden"][c:c + 2048].double(), s["labels"][c:c + 2048]
        keep = lab >= 0
        coef = torch.where(keep, s["scale"][c:c + 2048].double(), 0.0)
        lp = torch.log_softmax(h @ wt, dim=-1)
        rows = torch.arange(len(lab), device=w.device)
        lab = lab.clamp(min=0)
        loss -= (coef * lp[rows, lab]).sum()
        grad = lp.exp_()
        grad[rows, lab] -= 1.0
        grad *= coef[:, None]
        gh[c:c + 2048] = grad @ w
        gw += grad.t().contiguous() @ h
    return [loss, gh, gw]


_EXACT = {"attn": _exact_attn, "gdn": _exact_gdn, "prologue": _exact_prologue, "leafce": _exact_leafce}


def exact(case, seed):
    return _EXACT[case["op"]](case, seed)
