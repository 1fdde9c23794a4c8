# SPDX-License-Identifier: MIT
"""The workloads whose speed is measured, as cases that a timing program can
list, draw, prepare, run and check.

A case is a dict of plain values:

* ``kind``: ``decode`` (``decode`` of precomputed rows and ``backtrack``),
  ``train`` (``search``, ``losses.minimum_risk`` and the backward into the
  rows) or ``stepped`` (``beam_search`` over a step function);
* ``B, T, K, V``: examples, steps, beams, vocabulary;
* ``dtype`` (``f32``, ``f16``, ``bf16``) and ``logits`` (the rows are raw
  logits; otherwise log-probabilities);
* ``std``: the rows are drawn from N(0, std^2) (``zipf``: plus a bias of
  -1.1 ln(rank) shared by all rows; ``ties``: 5 % of the entries take one of 64
  values of their step), log-probabilities through a log-softmax;
* ``eos`` (-1: none; ``ends`` is added to its logit, so that beams finish),
  ``alpha``, ``min_length``, ``ngram``, ``rep``: the search's options;
* ``banned``: 1 % of the tokens are banned, per example; ``ragged``: each
  example has its own number of steps, from half of T to T.
"""

from __future__ import annotations

import math

import torch

import beamgrad_amd as bg

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}
_MOST = 4.9e9  # bytes of rows of the largest drawn case; the largest listed one holds 4.98e9


def _case(kind, B, T, K, V, dtype, logits, std, **more):
    case = dict(kind=kind, B=B, T=T, K=K, V=V, dtype=dtype, logits=logits, std=std, zipf=False, ties=False, eos=-1,
                ends=0.0, alpha=0.0, min_length=0, ngram=0, rep=1.0, banned=False, ragged=False)
    case.update(more)
    return case


def listed():
    cases = {
        # One prompt, a few beams, a short answer: an interactive call, where
        # the latency of the call itself is what its user sees.
        "one prompt": _case("decode", 1, 16, 4, 32000, "bf16", True, 3.0, eos=2, ends=9.0, alpha=0.6, min_length=2),
        # A small batch of log-probabilities in 32 bits (configuration C1).
        "small batch f32": _case("decode", 8, 32, 4, 32000, "f32", False, 2.0, eos=2, alpha=0.6),
        # A serving batch of a large vocabulary's raw logits (C2, the headline).
        "serving bf16 logits": _case("decode", 32, 64, 8, 151936, "bf16", True, 3.0, zipf=True, eos=151643,
                                     alpha=1.0, min_length=4),
        # Everything constrained, an odd vocabulary, ragged lengths (C3).
        "constrained f16": _case("decode", 64, 128, 5, 50257, "f16", False, 2.5, eos=50256, min_length=8, ngram=3,
                                 rep=1.2, banned=True, ragged=True),
        # Wide beams over rows with exact ties (C4).
        "wide beams f32": _case("decode", 16, 64, 64, 32000, "f32", False, 1.5, ties=True, eos=2, alpha=0.6),
        # A training step: minimum risk through the logits (C5).
        "train bf16 logits": _case("train", 16, 128, 8, 128256, "bf16", True, 3.0),
        # Logits kept in 32 bits, an odd vocabulary, beams that finish: the
        # 16 x 64 x 4 x 50k batch of the published benchmarks.
        "f32 logits odd": _case("decode", 16, 64, 4, 50257, "f32", True, 3.0, eos=50256, ends=7.0, alpha=0.6),
        # The same vocabulary in 16 bits: rows that start at odd elements.
        "bf16 logits odd": _case("decode", 32, 64, 5, 50257, "bf16", True, 3.0, eos=50256, ends=7.0, alpha=1.0,
                                 ragged=True),
        # Half-precision logits of a large vocabulary.
        "f16 logits": _case("decode", 8, 32, 8, 128256, "f16", True, 3.0, eos=128001, ends=7.0, alpha=1.0),
        # A training step on log-probabilities that a program's own
        # log-softmax made (16 x 64 x 4 x 50k, forward and backward).
        "train f32": _case("train", 16, 64, 4, 50000, "f32", False, 2.0, eos=2, ends=5.0, alpha=0.6),
        # A model in the loop: one engine call per step.
        "stepped f32": _case("stepped", 8, 24, 5, 32000, "f32", False, 2.5, eos=2, ends=5.0, alpha=0.6, min_length=4),
        # Very wide beams (4 x 8 x 256 x 32k of the published benchmarks).
        "256 beams f32": _case("decode", 4, 8, 256, 32000, "f32", False, 1.5, eos=2, alpha=0.6),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _spread(rng, low, high):
    """An integer of [low, high], spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["train"] * 3 + ["stepped"])
    dtype = rng.choice(["f32", "f16", "bf16", "bf16"])
    logits = kind != "stepped" and rng.random() < 0.6
    V = _spread(rng, 1000, 151936)
    if rng.random() < 0.5:  # vocabularies are often padded to a multiple of 8
        V += -V % 8
    K = _spread(rng, 1, 64)
    if kind == "decode" and rng.random() < 0.1:
        K = _spread(rng, 64, 256)
    T = _spread(rng, 4, 32 if kind == "stepped" else 128)
    B = _spread(rng, 1, 64)
    most = _MOST / (2.5 if kind == "train" else 4 if kind == "stepped" or K > 64 else 1)
    while B * T * K * V * _SIZE[dtype] > most:
        if B > 1 and (B >= T or T <= 4):
            B = B * 3 // 4
        elif T > 4:
            T = T * 3 // 4
        else:
            K = K * 3 // 4
    more = dict(alpha=rng.choice([0.0, 0.6, 1.0]))
    if rng.random() < 0.7:
        more.update(eos=rng.randrange(V), ends=rng.choice([0.0, 5.0, 7.0, 9.0]), min_length=rng.choice([0, 0, 2, 4]))
    if kind == "decode" and K <= 16 and rng.random() < 0.3:
        more.update(ngram=rng.choice([0, 2, 3]), rep=rng.choice([1.0, 1.2]), banned=rng.random() < 0.5)
    if kind != "stepped" and rng.random() < 0.3:
        more.update(ragged=True)
    return _case(kind, B, T, K, V, dtype, logits, rng.choice([1.5, 2.0, 3.0]), zipf=rng.random() < 0.25, **more)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _rows(case, gen):
    """The rows [B, T, K, V], one example at a time."""
    B, T, K, V = (case[d] for d in "BTKV")
    x = torch.empty(B, T, K, V, dtype=_TORCH[case["dtype"]], device="cuda")
    bias = None
    if case["zipf"]:
        rank = torch.randperm(V, generator=gen, device="cuda").to(torch.float32) + 1.0
        bias = -1.1 * torch.log(rank)
    for b in range(B):
        row = torch.randn(T, K, V, generator=gen, device="cuda").mul_(case["std"])
        if bias is not None:
            row += bias
        if case["eos"] >= 0 and case["ends"]:
            row[..., case["eos"]] += case["ends"]
        if not case["logits"]:
            row = torch.log_softmax(row, dim=-1)
        if case["ties"]:
            pool = row.reshape(T, -1)[:, :64].clone()
            tie = torch.rand(T, K, V, generator=gen, device="cuda") < 0.05
            pick = torch.randint(0, 64, (T, K, V), generator=gen, device="cuda")
            row = torch.where(tie, torch.gather(pool, 1, pick.reshape(T, -1)).reshape(T, K, V), row)
        x[b] = row
    return x


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, T, K, V = (case[d] for d in "BTKV")
    x = _rows(case, gen)
    steps = banned = costs = None
    if case["ragged"]:
        steps = torch.randint((T + 1) // 2, T + 1, (B,), generator=gen, device="cuda")
    if case["banned"]:
        banned = torch.zeros(B, V, dtype=torch.uint8, device="cuda")
        for b in range(B):
            banned[b, torch.randperm(V, generator=gen, device="cuda")[: V // 100]] = 1
    if case["kind"] == "train":
        costs = torch.rand(B, K, generator=gen, device="cuda")
    return x, steps, banned, costs


def prepare(case, seed):
    x, steps, banned, costs = _inputs(case, seed)
    options = bg.BeamOptions(beam_size=case["K"], eos_token=case["eos"],
                             min_length=case["min_length"], length_penalty_alpha=case["alpha"],
                             no_repeat_ngram_size=case["ngram"], repetition_penalty=case["rep"])
    state = dict(case=case, options=options, steps=steps, banned=banned, costs=costs)
    if case["kind"] == "stepped":
        # what the model would return at each step
        state["rows"] = [x[:, t].contiguous() for t in range(case["T"])]
    else:
        state["x"] = x.requires_grad_(case["kind"] == "train")
    return state


def run(state):
    case, options = state["case"], state["options"]
    if case["kind"] == "stepped":
        rows = state["rows"]
        with torch.no_grad():
            result = bg.beam_search(lambda beams: rows[beams.step], options, case["T"], batch_size=case["B"],
                                    device="cuda")
        return [result.scores, result.raw_scores, result.lengths, result.sequences]
    if case["kind"] == "train":
        x = state["x"]
        x.grad = None
        result = bg.search(x, options, state["steps"], from_logits=case["logits"], banned_mask=state["banned"])
        loss = bg.losses.minimum_risk(result, state["costs"])
        loss.backward()
        return [result.scores.detach(), result.raw_scores.detach(), result.lengths, result.sequences, loss.detach(),
                x.grad]
    out = bg.decode(state["x"], options, state["steps"], from_logits=case["logits"], banned_mask=state["banned"])
    return [*out[:9], bg.backtrack(out)]


def work(case):
    """Every row that a search without finished beams reads, once; a training
    step also writes the rows' gradient and, from logits, reads one row per
    example and step again for its softmax. One operation per entry read, and
    two more for a logsumexp's term."""
    B, T, K, V = (case[d] for d in "BTKV")
    steps = T * (0.75 if case["ragged"] else 1.0)
    entries = B * (1 + (steps - 1) * K) * V
    moved = entries
    if case["kind"] == "train":
        moved += B * T * K * V + (B * steps * V if case["logits"] else 0)
    return {"bytes": moved * _SIZE[case["dtype"]], "flops": entries * (3 if case["logits"] else 1)}


def tolerance(case):
    """The results are a given sequence of single rounded operations for every
    input (the reference library's bits are part of the interface), so another
    correct implementation gives the same ones."""
    return "exact"


# ---------------------------------------------------------------------------
# The same results in plain torch, in 64 bits
# ---------------------------------------------------------------------------


def _ordered(x):
    """float32 as an int64 that sorts like it, -0 with +0."""
    u = x.contiguous().view(torch.int32).long()
    return torch.where(u >= 0, u, -(u & 0x7FFFFFFF))


def _penalty(length, alpha):
    return ((5.0 + length.clamp(min=1).double()) / 6.0) ** alpha


def _allowed(case, banned, prefix, plen, length):
    """Which tokens each beam may take [B, K, V], and which are in its prefix."""
    B, K, T = prefix.shape
    V, n = case["V"], case["ngram"]
    ok = torch.ones(B, K, V, dtype=torch.bool, device="cuda")
    seen = torch.zeros(B, K, V + 1, dtype=torch.bool, device="cuda")
    if banned is not None:
        ok &= banned[:, None, :].eq(0)
    if case["eos"] >= 0 and case["min_length"]:
        ok[:, :, case["eos"]] &= length + 1 >= case["min_length"]
    at = torch.arange(T, device="cuda")
    if case["rep"] > 1.0:
        seen.scatter_(2, torch.where(at < plen[..., None], prefix, V), True)
    if n > 1 and T >= n:
        gram = prefix.unfold(2, n, 1)  # [B, K, T - n + 1, n]
        tail = prefix.gather(2, (plen[..., None] - (n - 1) + at[: n - 1]).clamp(min=0))
        hit = (gram[..., : n - 1] == tail[:, :, None, :]).all(-1) & (at[: T - n + 1] + n <= plen[..., None])
        blocked = torch.zeros(B, K, V + 1, dtype=torch.bool, device="cuda")
        blocked.scatter_(2, torch.where(hit, gram[..., n - 1], V), True)
        ok &= ~blocked[..., :V]
    return ok, seen[..., :V]


def _search64(case, x, steps, banned):
    """The search: candidates ranked by their scores as the search keeps them
    (32-bit sums, ties by raw score, parent and token), values in 64 bits."""
    B, T, K, V = (case[d] for d in "BTKV")
    dev, inf = "cuda", float("inf")
    raw32 = torch.full((B, K), -inf, device=dev)
    raw32[:, 0] = 0.0
    raw, score = raw32.double(), raw32.double()
    length = torch.zeros(B, K, dtype=torch.long, device=dev)
    last = torch.full((B, K), -1, dtype=torch.long, device=dev)
    done = torch.zeros(B, K, dtype=torch.bool, device=dev)
    prefix = torch.full((B, K, T), -1, dtype=torch.long, device=dev)
    plen = torch.zeros(B, K, dtype=torch.long, device=dev)
    limited = banned is not None or case["ngram"] > 1 or case["rep"] > 1.0 or (case["eos"] >= 0 and case["min_length"])
    log_rep = math.log(case["rep"])
    every = torch.arange(B, device=dev)[:, None]
    trace = {k: [] for k in ("score", "raw", "parent", "token", "grown", "lse")}
    for t in range(T):
        rows = x[:, t].float()
        lse = torch.zeros(B, K, dtype=torch.float64, device=dev)
        if case["logits"]:
            lse = torch.logsumexp(rows.double(), -1)
            rows = rows - lse.float()[..., None]
        if limited:
            ok, seen = _allowed(case, banned, prefix, plen, length)
            if case["rep"] > 1.0:
                rows = torch.where(seen, rows - torch.tensor(log_rep, dtype=torch.float32, device=dev), rows)
            rows = rows.masked_fill(~ok, -inf)
        cand = rows.add_(raw32[..., None]) if case["logits"] or limited else rows + raw32[..., None]
        factor = 1.0 / _penalty(length + 1, case["alpha"]).float()
        ranked = cand * factor[..., None]
        if done.any():  # a finished beam is one candidate: itself
            cand[done], ranked[done] = -inf, -inf
            b, k = done.nonzero(as_tuple=True)
            cand[b, k, last[b, k]] = raw32[b, k]
            ranked[b, k, last[b, k]] = raw32[b, k] / _penalty(length[b, k], case["alpha"]).float()
        key = (_ordered(ranked) * 2**32 + _ordered(cand) + 2**31).reshape(B, K * V)
        n = min(K, K * V)
        least = torch.topk(key, n).values[:, -1:]
        b, i = (key >= least).nonzero(as_tuple=True)  # by example, then by (parent, token)
        order = torch.sort(key[b, i], descending=True, stable=True).indices
        order = order[torch.sort(b[order], stable=True).indices]
        b, i = b[order], i[order]
        first = torch.searchsorted(b, torch.arange(B, device=dev))
        at = i[first[:, None] + torch.arange(n, device=dev)]
        parent, token = at // V, at % V
        chosen32 = cand.reshape(B, K * V).gather(1, at)
        live = chosen32 > -inf
        grown = live & ~done.gather(1, parent)
        value = x[every, t, parent, token].double() - lse.gather(1, parent)
        if case["rep"] > 1.0:
            value = value - log_rep * seen[every, parent, token]
        on = (t < steps)[:, None].expand(B, K)
        parent, token = torch.where(live, parent, -1), torch.where(live, token, -1)
        p = parent.clamp(min=0)
        new_raw = raw.gather(1, p) + torch.where(grown, value, 0.0)
        new_raw = new_raw.masked_fill(~live, -inf)
        new_length = torch.where(live, length.gather(1, p) + grown, 0)
        new_done = live & (done.gather(1, p) | (token == case["eos"])) if case["eos"] >= 0 else torch.zeros_like(done)
        new_score = new_raw / _penalty(new_length, case["alpha"])
        new_prefix, new_plen = prefix[every, p], plen.gather(1, p)
        e, k = (on & grown).nonzero(as_tuple=True)
        new_prefix[e, k, new_plen[e, k]] = token[e, k]
        for name, v in (("score", new_score), ("raw", new_raw)):
            trace[name].append(v.masked_fill(~on, -inf))
        for name, v in (("parent", parent), ("token", token)):
            trace[name].append(v.masked_fill(~on, -1))
        trace["grown"].append(grown & on)
        trace["lse"].append(lse)
        raw32, raw, score = torch.where(on, chosen32, raw32), torch.where(on, new_raw, raw), torch.where(on, new_score, score)
        length, last, done = torch.where(on, new_length, length), torch.where(on, token, last), torch.where(on, new_done, done)
        prefix, plen = torch.where(on[..., None], new_prefix, prefix), torch.where(on, new_plen + grown, plen)
    return score, raw, length, trace


def exact(case, seed):
    x, steps, banned, costs = _inputs(case, seed)
    B, T, K, V = (case[d] for d in "BTKV")
    if steps is None:
        steps = torch.full((B,), T, device="cuda")
    score, raw, length, trace = _search64(case, x, steps, banned)
    if case["kind"] == "stepped":
        return [score, raw, None, None]
    if case["kind"] == "decode":
        return [score, raw, None, None, None, None, torch.stack(trace["score"], 1), torch.stack(trace["raw"], 1), None,
                None]
    live = torch.isfinite(score)
    p = torch.softmax(score, -1)
    cost = torch.where(live, costs.double(), 0.0)
    risk = (p * cost).sum(-1)
    g = p * (cost - risk[:, None]) / B / _penalty(length, case["alpha"])  # of the raw scores
    g = torch.where(live, g, 0.0)
    grad = torch.zeros(B, T, K, V, dtype=torch.float64, device="cuda")
    every = torch.arange(B, device="cuda")[:, None].expand(B, K)
    for t in reversed(range(T)):
        parent, token, grown = (trace[k][t] for k in ("parent", "token", "grown"))
        on = (t < steps)[:, None]
        at = parent.clamp(min=0)
        entry = torch.where(grown, g, 0.0)
        if case["logits"]:
            total = torch.zeros(B, K, dtype=torch.float64, device="cuda").scatter_add_(1, at, entry)
            b, k = torch.zeros(B, K, dtype=torch.bool, device="cuda").scatter_(1, at, grown).nonzero(as_tuple=True)
            soft = torch.exp(x[b, t, k].double() - trace["lse"][t][b, k, None])
            grad[b, t, k] = -soft * total[b, k, None]
        grad.index_put_((every, torch.full_like(at, t), at, token.clamp(min=0)), entry, accumulate=True)
        up = torch.zeros_like(g).scatter_add_(1, at, torch.where(parent >= 0, g, 0.0))
        g = torch.where(on, up, g)
    return [score, raw, None, None, risk.mean(), grad]
