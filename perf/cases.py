"""What a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``op`` names the call:

* ``layer``   -- ``attention_matrix(q, kp, vp, prepared)``: one decode-step attention layer on
  resident K/V pools under a plan that the program keeps for all layers and steps;
* ``pack``    -- ``attention(q, k, v, prepared)``: the same from token-major K and V, packed
  into the pool layouts by the call;
* ``decode``  -- one layer's attention block of a decode step: ``decode_append`` (RoPE, the
  scatter of the step's K/V into the pools, the Q layout), then ``attention_matrix`` under a
  ``CachedDecodePlan``; with ``update`` the step also sets the tails' lengths first, as it
  does once per step;
* ``replan``  -- ``schedule``, ``prepare`` and one ``attention_matrix``: what a step costs when
  the tree has changed (requests came or went, or an uncached decoder);
* ``model``   -- one ``CachedPrefixDecoder.step`` of a Qwen3-shaped model, replayed from a HIP
  graph, which returns the logits; the token is taken back first, as a program does that
  rejects a drafted token, so that every pass decodes the same step.

The prefix tree is given by ``tree`` (levels of shared nodes, root first: "2048/64*4" is a
2048-token root with four 64-token children), ``requests`` spread evenly over the last level,
and a private part of ``private + vary * r`` tokens for request ``r``.  ``inner`` requests end
at the first node of the second level, ``dup`` requests repeat the first requests' paths.
The pools hold the tree's tokens, the decode tails and ``pad`` unused positions; nothing
rounds their capacity up, as nothing does when a program packs the K/V it has.
"""
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tree-attention-scheduling_amd"))

from tree_attention import CostModel, KVTree, schedule  # noqa: E402
from tree_attention.kernels import (CachedDecodePlan, attention, attention_matrix, decode_append,  # noqa: E402
                                    prepare as prepare_plan)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BASE = dict(op="layer", tree="1024", requests=8, private=64, vary=0, inner=0, dup=0, pad=0, hq=32, hk=8, d=128,
            dtype="bf16", method="cube", tail=0, generated=0, update=False, layers=0)


def _case(name, **kw):
    return {"name": name, **BASE, **kw}


def listed():
    return [
        # a small batch over one system prompt: the smallest call, where latency and launches count
        _case("small_8x1088", tree="1024", requests=8, private=64),
        # a small model's heads (8 query / 2 KV, head dim 64) in fp16 over a ragged batch, whose
        # pools hold exactly the tree's 1745 tokens
        _case("ragged_d64_fp16", tree="257", requests=32, private=31, vary=1, hq=8, hk=2, d=64, dtype="fp16"),
        # medium contexts of which a quarter is private, two levels of sharing
        _case("grid_32x4096_fp16", tree="1536/1536*2", requests=32, private=1024, dtype="fp16"),
        # few-shot prompts under one instruction: three levels, a request at an inner node, duplicates
        _case("nested_35", tree="4096/1024*8/256*4", requests=32, private=0, inner=1, dup=2),
        # two branches of unequal conversations, pools of an odd number of tokens
        _case("branches_odd_24", tree="768/384*2", requests=24, private=192, vary=17, pad=3),
        # the benchmark's layer: 128 requests over one long shared document
        _case("headline_128x8192", tree="8128", requests=128, private=64),
        # the largest call: nothing shared, memory bound (4.3 GB of K/V)
        _case("private_128x8192", tree="0", requests=128, private=8192),
        # K/V straight from a prefill, token-major, ragged private parts
        _case("pack_unequal_32", op="pack", tree="1024", requests=32, private=32, vary=31),
        # one layer's attention block in a decode step of the Qwen3-4B-shaped workload
        _case("decode_block_32x2240", op="decode", tree="2048/64*4", requests=32, private=128, tail=16, generated=8),
        # the cached-plan protocol: set the tails' lengths, then one layer
        _case("protocol_step_32x1088", op="decode", tree="1024", requests=32, private=64, tail=16, generated=8,
              update=True),
        # the tree has changed: plan, lower and attend
        _case("replan_32x1088", op="replan", tree="1024", requests=32, private=64),
        # a whole decode step of a Qwen3-4B-shaped model (two layers, the vocabulary in full)
        _case("model_step_32x2240", op="model", tree="2048/64*4", requests=32, private=128, tail=4, generated=1,
              layers=2),
    ]


def draw(rng):
    """One more layer, decode block or re-planned step from the ranges above."""
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    while True:
        d = rng.choice((128, 128, 128, 64, 64, 32))
        hq, hk = rng.choice({128: ((32, 8), (32, 8), (16, 8), (64, 8)), 64: ((8, 2), (32, 8), (16, 2)),
                             32: ((8, 2), (4, 2), (8, 8))}[d])
        requests, context = log_int(4, 128), log_int(96, 8192)
        shared = 0 if rng.random() < 0.15 else int(context * rng.uniform(0.2, 0.99))
        depth = rng.choice((1, 1, 2, 3)) if shared >= 64 else 1
        cuts = sorted(rng.sample(range(1, shared), depth - 1)) if depth > 1 else []
        lens = [b - a for a, b in zip([0] + cuts, cuts + [shared])]
        tree = "/".join(f"{n}*{rng.choice((2, 3, 4))}" if i else str(n) for i, n in enumerate(lens))
        op = rng.choice(("layer", "layer", "layer", "layer", "decode", "decode", "replan"))
        case = dict(BASE, op=op, tree=tree, requests=requests, private=max(1, context - shared),
                    vary=rng.choice((0, 0, 1, 3, 7)), hq=hq, hk=hk, d=d, dtype=rng.choice(("bf16", "bf16", "fp16")),
                    method=rng.choice(("cube", "cube", "cube", "greedy", "fixed", "request")), pad=rng.randrange(8))
        if op == "decode":  # a decoder's pools: capacity rounded up to whole 8-token groups
            tail = log_int(4, 64)
            case.update(tail=tail, generated=rng.randint(1, tail), update=rng.random() < 0.3)
            case["pad"] = -(_tokens(case) + requests * tail) % 8
        # at most half the largest listed layer's K/V, and re-planned trees of a serving batch
        if _capacity(case) * hk * d <= 1 << 29 and (op != "replan" or requests * context <= 1 << 17):
            return case


# ---------------------------------------------------------------- the tree of a case
def _spec(case):
    """(parents, lengths, terminals) of the case's tree, nodes in depth-first order."""
    levels = [(int(n), int(m or 1)) for n, _, m in (part.partition("*") for part in case["tree"].split("/"))]
    leaves = 1
    for _, width in levels[1:]:
        leaves *= width
    per_leaf = [[] for _ in range(leaves)]
    for r in range(case["requests"]):
        per_leaf[r * leaves // case["requests"]].append(r)
    parents, lengths, ends, second = [], [], {}, 0
    seen = 0

    def grow(parent, depth):
        nonlocal seen, second
        below = 1
        for _, width in levels[depth + 1:]:
            below *= width
        if not any(per_leaf[seen:seen + below]):  # no request comes through here: no such node
            seen += below
            return
        node = len(parents)
        parents.append(parent)
        lengths.append(levels[depth][0])
        if depth == 1 and not second:
            second = node
        if depth + 1 < len(levels):
            for _ in range(levels[depth + 1][1]):
                grow(node, depth + 1)
            return
        for r in per_leaf[seen]:
            private = case["private"] + case["vary"] * r
            if private == 0:
                ends[r] = node
                continue
            ends[r] = len(parents)
            parents.append(node)
            lengths.append(private)
        seen += 1

    grow(-1, 0)
    terminals = [ends[r] for r in range(case["requests"])]
    return parents, lengths, terminals + [second] * case["inner"] + terminals[:case["dup"]]


def _tokens(case):
    return sum(_spec(case)[1])


def _capacity(case):
    reserved = len(_spec(case)[2]) * case["tail"] if case["op"] in ("decode", "model") else 0
    return _tokens(case) + reserved + (case["pad"] if case["op"] != "pack" else 0)


def _paths(case):
    """Every request's runs of physical tokens, the decode tail's included."""
    parents, lengths, terminals = _spec(case)
    starts = [0]
    for n in lengths:
        starts.append(starts[-1] + n)
    paths = []
    for r, node in enumerate(terminals):
        runs = []
        while node >= 0:
            runs.append((starts[node], starts[node] + lengths[node]))
            node = parents[node]
        if case["op"] == "decode":
            t0 = starts[-1] + r * case["tail"]
            runs.insert(0, (t0, t0 + case["generated"]))
        paths.append([run for run in reversed(runs) if run[1] > run[0]])
    return paths


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    dev, dtype = torch.device("cuda:0"), DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)
    hq, hk, d, cap = case["hq"], case["hk"], case["d"], _capacity(case)
    nreq = len(_spec(case)[2])

    def randn(*shape):
        return torch.randn(shape, generator=g, device=dev, dtype=dtype)

    x = {}
    if case["op"] == "pack":
        x.update(q=randn(nreq, hq, d), k=randn(cap, hk, d), v=randn(cap, hk, d))
    elif case["op"] == "decode":
        x.update(kp=randn(hk, d, cap), vp=randn(hk, cap, d), q=randn(nreq, 1, hq, d), k=randn(nreq, 1, hk, d),
                 v=randn(nreq, 1, hk, d))
        base = _tokens(case)
        where = [base + r * case["tail"] + case["generated"] - 1 for r in range(nreq)]
        x["slots"] = torch.tensor(where, device=dev, dtype=torch.int32)
        length = torch.tensor([sum(b - a for a, b in runs) - 1 for runs in _paths(case)], device=dev)
        inv = 1.0 / (1e6 ** (torch.arange(0, d, 2, device=dev, dtype=torch.float32) / d))
        angle = torch.cat([length[:, None] * inv] * 2, dim=-1)[:, None]
        x.update(cos=angle.cos().to(dtype), sin=angle.sin().to(dtype))
    else:
        x.update(q=randn(nreq, hq, d), kp=randn(hk, d, cap), vp=randn(hk, cap, d))
    return x


def prepare(case, seed):
    if case["op"] == "model":
        return _prepare_model(case, seed)
    s = dict(_inputs(case, seed), op=case["op"], update=case["update"], generated=case["generated"])
    tree = KVTree.synthetic(*_spec(case))
    heads = (case["hq"], case["hk"], case["d"])
    plan_args = (tree, *heads, case["method"], CostModel.mi355x())
    if case["op"] == "replan":
        s["plan_args"] = plan_args
        return s
    plan = schedule(*plan_args)
    if case["op"] == "decode":
        shape_of_q = torch.empty((s["q"].shape[0], heads[0], heads[2]), device=s["q"].device, dtype=s["q"].dtype)
        s["cached"] = CachedDecodePlan(plan, shape_of_q, tree.storage_tokens, case["tail"])
        s["prepared"] = s["cached"].update(case["generated"])
    else:
        s["prepared"] = prepare_plan(plan, s["q"])
    return s


def _prepare_model(case, seed):
    from tree_attention.benchmark_decode import _model
    from tree_attention.qwen import CachedPrefixDecoder

    dev = torch.device("cuda:0")
    model = _model(case["layers"], dev)
    g = torch.Generator().manual_seed(seed)
    parents, lengths, terminals = _spec(case)
    # the node's index leads its tokens, so that no two siblings start alike
    ids = [[10 + i] + torch.randint(1000, 151_936, (n - 1,), generator=g).tolist() for i, n in enumerate(lengths)]

    def path(node):
        return [] if node < 0 else path(parents[node]) + ids[node]

    decoder = CachedPrefixDecoder(model, [path(t) for t in terminals], case["tail"], case["method"],
                                  CostModel.mi355x(), prefill="tree", graph=True)
    tokens = torch.randint(1000, 151_936, (len(terminals),), generator=g).tolist()
    decoder.step(tokens)  # the first step captures the graph that later ones replay
    return {"op": "model", "decoder": decoder, "tokens": tokens}


def run(state):
    op = state["op"]
    if op == "layer":
        return attention_matrix(state["q"], state["kp"], state["vp"], state["prepared"])
    if op == "pack":
        return attention(state["q"], state["k"], state["v"], state["prepared"])
    if op == "replan":
        prepared = prepare_plan(schedule(*state["plan_args"]), state["q"])
        return attention_matrix(state["q"], state["kp"], state["vp"], prepared)
    if op == "decode":
        kp, vp = state["kp"], state["vp"]
        prepared = state["cached"].update(state["generated"]) if state["update"] else state["prepared"]
        q = decode_append(state["q"], state["k"], state["v"], state["cos"], state["sin"], state["slots"], kp, vp)
        return {"out": attention_matrix(q, kp, vp, prepared), "kp": kp, "vp": vp}
    decoder = state["decoder"]
    for seq in decoder.sequences:  # take the token back
        seq.pop()
    decoder.generated -= 1
    decoder.used -= len(decoder.sequences)
    return decoder.step(state["tokens"])


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    hq, hk, d = case["hq"], case["hk"], case["d"]
    paths = _paths(case)
    nreq = len(paths)
    read = sum({run: run[1] - run[0] for runs in paths for run in runs}.values())
    logical = sum(b - a for runs in paths for a, b in runs)
    nbytes = 2 * (2 * read * hk * d + 2 * nreq * hq * d)
    flops = 4 * logical * hq * d
    if case["op"] == "decode":  # the step's K and V in and into the pools, RoPE's tables
        nbytes += 2 * nreq * d * (4 * hk + 2)
    if case["op"] == "model":
        # Qwen3-4B-shaped layers (hidden 2560, FFN 9728) and the 151,936-row head: weights once
        layer = 2560 * (hq + 2 * hk) * d + hq * d * 2560 + 3 * 2560 * 9728
        weights = case["layers"] * layer + 151_936 * 2560
        logits = nreq * 151_936
        logical += nreq * case["generated"]
        return {"bytes": case["layers"] * nbytes + 2 * weights + 2 * logits,
                "flops": case["layers"] * 4 * logical * hq * d + 2 * nreq * weights}
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16: the probabilities and the output are rounded to 8 bits (0.24 % of the output's norm
    # against 64 bits); fp16: to 11 bits.  The limits are four times what the same layers showed
    # under plans that sum in another order (bf16: 0.31 % and 0.014; fp16: 0.046 % and 0.002 of
    # the root mean square).  A whole model adds its own roundings (1.1 % between two plans).
    if case["op"] == "model":
        return {"rel": 0.03}
    return {"rel": 1.2e-2, "max": 0.08} if case["dtype"] == "bf16" else {"rel": 2e-3, "max": 0.02}


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    if case["op"] == "model":
        return None
    x = _inputs(case, seed)
    hq, hk, d = case["hq"], case["hk"], case["d"]
    q = x["q"].double().reshape(-1, hq, d)
    extra = {}
    if case["op"] == "pack":
        kp, vp = x["k"].permute(1, 2, 0).contiguous(), x["v"].permute(1, 0, 2).contiguous()
    elif case["op"] == "decode":
        def rope(t):
            half = torch.cat((-t[..., d // 2:], t[..., :d // 2]), dim=-1)
            return t * x["cos"].double() + half * x["sin"].double()

        where = x["slots"].long()
        q = rope(x["q"][:, 0].double())
        kp, vp = x["kp"].double(), x["vp"].double()
        kp.index_copy_(2, where, rope(x["k"][:, 0].double()).permute(1, 2, 0))
        vp.index_copy_(1, where, x["v"][:, 0].double().permute(1, 0, 2))
        extra = {"kp": kp, "vp": vp}
    else:
        kp, vp = x["kp"], x["vp"]
    out = torch.empty_like(q)
    for r, runs in enumerate(_paths(case)):
        k = torch.cat([kp[:, :, a:b] for a, b in runs], dim=2).double()
        v = torch.cat([vp[:, a:b] for a, b in runs], dim=1).double()
        s = torch.bmm(q[r].reshape(hk, hq // hk, d), k) / d ** 0.5
        out[r] = torch.bmm(torch.softmax(s, dim=-1), v).reshape(hq, d)
    return {"out": out, **extra} if extra else out
