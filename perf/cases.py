"""The work that programs have this framework do, as cases for timing and comparing builds.

Rollout (sampling of one decode step's logits), scoring (log-probs of given tokens from hidden
states and the head's weight), learning (the same with its backward) and the loss over a batch
of responses, each through the package's public functions with their default checks.  Sizes are
the benchmark configurations' (``dsv41_rocm.workloads``) and the ranges around them.

``listed()`` are fixed cases, ``draw(rng)`` gives further ones from the same ranges,
``prepare(case, seed)`` the inputs, ``run(state)`` one pass, ``work(case)`` what a pass cannot do
without, ``tolerance(case)`` and ``exact(case, seed)`` how its outputs compare.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.add_paths()

import dsv41_rocm  # noqa: E402

DEV = "cuda"
NO_KNOBS = {"temperature": 1.0, "repetition_penalty": 1.0, "presence_penalty": 0.0, "frequency_penalty": 0.0,
            "top_k": 0, "top_p": 1.0, "min_p": 0.0, "greedy": False}


def _sample(rows, vocab, dtype, history=0, stride=None, **knobs):
    return {"kind": "sample", "rows": rows, "vocab": vocab, "stride": stride or vocab, "dtype": dtype,
            "history": history, **{**NO_KNOBS, **knobs}}


def listed():
    return [
        # one token of an autoregressive decode: the smallest call there is
        {"name": "decode_token", "kind": "next", "vocab": 151936, "dtype": "f32", "temperature": 0.7},
        # a prompt group's decode step with the usual serving knobs (benchmark configuration A)
        {"name": "group_topk_8", **_sample(8, 129280, "f32", 256, temperature=0.7, repetition_penalty=1.1, top_k=50,
                                           top_p=0.95)},
        # nucleus sampling of a decode batch, logits a view of a head padded to a multiple of 128
        {"name": "nucleus_48", **_sample(48, 151851, "bf16", stride=151936, temperature=0.8, top_p=0.9)},
        # penalized full-vocabulary sampling (benchmark configuration B)
        {"name": "penalized_256", **_sample(256, 151936, "bf16", 2048, presence_penalty=0.5, frequency_penalty=0.2)},
        # the training default, no truncation and no penalties, over a ragged number of live rows
        {"name": "train_rollout_1000", **_sample(1000, 129280, "f32", temperature=1.0)},
        # every knob on, the largest batch (benchmark configuration E)
        {"name": "all_knobs_4096", **_sample(4096, 151936, "f32", 4096, temperature=0.6, repetition_penalty=1.05,
                                             top_k=1024, top_p=0.98, min_p=0.05)},
        # behaviour log-probs of one response replayed from its logits
        {"name": "replay_300", "kind": "replay", "rows": 300, "vocab": 151936, "stride": 151936, "dtype": "bf16",
         "history": 0, **{**NO_KNOBS, "temperature": 0.7}},
        # one response scored by the large head
        {"name": "score_response_331", "kind": "score", "tokens": 331, "hidden": 7168, "vocab": 129280,
         "temperature": 1.0, "ratio": False},
        # the response tokens of a padded batch scored by the small head
        {"name": "score_masked_8x1024", "kind": "masked", "batch": 8, "length": 1024, "hidden": 2048, "vocab": 151936,
         "temperature": 0.8},
        # a microbatch scored with its importance weights (benchmark configuration D)
        {"name": "score_ratio_16384", "kind": "score", "tokens": 16384, "hidden": 7168, "vocab": 129280,
         "temperature": 1.0, "ratio": True},
        # the learner's chunk of 2048 tokens: forward and both gradients
        {"name": "learn_chunk_2048", "kind": "learn", "tokens": 2048, "hidden": 7168, "vocab": 129280,
         "temperature": 1.0, "weight_grad": True},
        # the loss over a batch of ragged responses, its metrics and its gradient
        {"name": "tis_loss_32", "kind": "loss", "loss": "tis", "responses": 32, "longest": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng):
    return rng.choice([129280, 151936, 151936, _log_int(rng, 8192, 151936)])


def draw(rng):
    kind = rng.choice(["next"] + ["sample"] * 5 + ["replay"] + ["score"] * 3 + ["masked", "learn", "learn", "loss"])
    temperature = rng.choice([1.0, 0.6, 0.7, round(rng.uniform(0.3, 1.5), 3)])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "next":
        return {"kind": kind, "vocab": _vocab(rng), "dtype": dtype, "temperature": temperature}
    if kind in ("sample", "replay"):
        rows, vocab = _log_int(rng, 1, 4096), _vocab(rng)
        case = _sample(rows, vocab, dtype, stride=(vocab + 127) // 128 * 128, temperature=temperature)
        mode = rng.choice(["full", "topk", "topk_topp", "topp", "minp", "all", "greedy"])
        if kind == "replay":
            case["kind"], mode = "replay", "full"
        if mode in ("topk", "topk_topp", "all"):
            case["top_k"] = rng.choice([20, 50, 1024]) if mode != "all" else 1024
        if mode in ("topk_topp", "topp", "all"):
            case["top_p"] = rng.choice([0.8, 0.9, 0.95, 0.98])
        if mode in ("minp", "all"):
            case["min_p"] = rng.choice([0.02, 0.05, 0.1])
        case["greedy"] = mode == "greedy"
        if rng.random() < 0.5:
            case["history"] = _log_int(rng, 16, 4096)
            if rng.random() < 0.5:
                case["repetition_penalty"] = rng.choice([1.05, 1.1])
            else:
                case["presence_penalty"], case["frequency_penalty"] = 0.5, 0.2
        return case
    if kind == "loss":
        return {"kind": kind, "loss": rng.choice(["tis", "grpo", "grpo_kl"]), "responses": _log_int(rng, 1, 256),
                "longest": _log_int(rng, 64, 8192)}
    hidden, vocab = rng.choice([(2048, 151936), (7168, 129280), (8 * _log_int(rng, 64, 896), _vocab(rng))])
    most = 3.0e13 / (2.0 * hidden * vocab)  # tokens of the largest listed case's operations
    if kind == "learn":
        return {"kind": kind, "tokens": _log_int(rng, 1, int(min(16384, most / 3))), "hidden": hidden, "vocab": vocab,
                "temperature": temperature, "weight_grad": rng.random() < 0.5}
    if kind == "masked":
        batch = rng.choice([1, 4, 8, 16])
        return {"kind": kind, "batch": batch, "length": _log_int(rng, 32, 16384 // batch), "hidden": hidden,
                "vocab": vocab, "temperature": temperature}
    return {"kind": kind, "tokens": _log_int(rng, 1, int(min(16384, most))), "hidden": hidden, "vocab": vocab,
            "temperature": temperature, "ratio": rng.random() < 0.5}


# ------------------------------------------------------------------------------------- inputs
def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(seed)


def _logits(case, rows, g):
    """Next-token logits with a Zipf-like head, N(0, 1) - 1.1 log(rank), the ranks in an order of
    each row's own; the rows' id of each rank comes along (for histories of likely tokens)."""
    V, stride = case["vocab"], case.get("stride", case["vocab"])
    order = torch.randperm(V, generator=g, device=DEV)  # order[j] = rank - 1 of position j
    place = torch.empty_like(order)
    place[order] = torch.arange(V, device=DEV)
    bias = -1.1 * torch.log((order + 1).float())
    shift = torch.randint(0, V, (rows,), generator=g, device=DEV)
    out = torch.empty(rows, stride, dtype=torch.float32 if case["dtype"] == "f32" else torch.bfloat16, device=DEV)
    ids = torch.arange(V, device=DEV)
    for r in range(0, rows, 256):
        e = min(rows, r + 256)
        noise = torch.randn(e - r, V, generator=g, device=DEV)
        out[r:e, :V] = noise + bias[(ids[None, :] + shift[r:e, None]) % V]
        out[r:e, V:] = 0

    def likely(n):  # ids whose ranks follow 1 / rank, so likely ones repeat
        rank = torch.pow(float(V), torch.rand(rows, n, generator=g, device=DEV)).long().clamp_(1, V)
        return (place[rank - 1] - shift[:, None]) % V

    return out[:, :V], likely


def _head(case, g, tokens):
    H, V = case["hidden"], case["vocab"]
    x = torch.randn(tokens, H, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.empty(V, H, dtype=torch.bfloat16, device=DEV)
    for r in range(0, V, 16384):
        e = min(V, r + 16384)
        w[r:e] = 0.02 * torch.randn(e - r, H, generator=g, device=DEV)
    return x, w, torch.randint(0, V, (tokens,), generator=g, device=DEV)


def _lengths(case):
    """Ragged response lengths, a few of them the longest allowed, as sampled responses have."""
    n = case["responses"]
    r = np.random.RandomState(n)
    return [int(v) for v in np.clip(np.round(case["longest"] * r.beta(1.2, 2.0, n) * 1.3), 1, case["longest"])]


def _knobs(case):
    return {k: case[k] for k in NO_KNOBS if k != "greedy"}


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "next":
        logits, _ = _logits(case, 1, g)
        return {"kind": kind, "logits": logits, "temperature": case["temperature"], "generator": _gen(seed, "cpu")}
    if kind in ("sample", "replay"):
        logits, likely = _logits(case, case["rows"], g)
        state = {"kind": kind, "logits": logits, "knobs": _knobs(case), "greedy": case["greedy"],
                 "history": likely(case["history"]) if case["history"] else None}
        if kind == "sample":
            state["uniforms"] = torch.rand(case["rows"], generator=g, device=DEV)
        else:
            state["ids"] = likely(1).reshape(-1)
            for k in ("top_k", "top_p", "min_p"):
                state["knobs"].pop(k)
        return state
    if kind == "loss":
        lengths = _lengths(case)
        n = sum(lengths)
        behavior = -torch.empty(n, device=DEV).exponential_(1.2, generator=g)
        old = (behavior + 0.15 * torch.randn(n, generator=g, device=DEV)).clamp_(max=0.0)
        cur = (old + 0.1 * torch.randn(n, generator=g, device=DEV)).clamp_(max=0.0)
        ref = (old + 0.1 * torch.randn(n, generator=g, device=DEV)).clamp_(max=0.0)
        return {"kind": kind, "loss": case["loss"], "lengths": lengths, "current": cur.requires_grad_(),
                "old": list(old.split(lengths)), "behavior": list(behavior.split(lengths)),
                "reference": list(ref.split(lengths)),
                "advantages": torch.randn(len(lengths), generator=_gen(seed, "cpu"))}
    if kind == "masked":
        B, L = case["batch"], case["length"]
        x, w, targets = _head(case, g, B * L)
        # one span per row: the response after its prompt, up to its own end
        r = np.random.RandomState(seed % (1 << 31))
        begin = torch.tensor((L * r.uniform(0.05, 0.4, B)).astype("int64"), device=DEV)[:, None]
        end = torch.tensor(np.maximum((L * r.uniform(0.6, 1.0, B)).astype("int64"), 1), device=DEV)[:, None]
        at = torch.arange(L, device=DEV)[None, :]
        return {"kind": kind, "hidden": x.view(B, L, -1), "weight": w, "targets": targets.view(B, L),
                "mask": (at >= begin) & (at < end), "temperature": case["temperature"]}
    x, w, targets = _head(case, g, case["tokens"])
    state = {"kind": kind, "hidden": x, "weight": w, "targets": targets, "temperature": case["temperature"],
             "behavior": None}
    if kind == "learn":
        x.requires_grad_()
        w.requires_grad_(case["weight_grad"])
        n = case["tokens"]
        state["grads"] = (torch.randn(n, generator=g, device=DEV) / n, torch.full((n,), -0.01 / n, device=DEV))
    elif case["ratio"]:
        # what an earlier policy reported for these tokens: about log(1 / V) under random weights
        state["behavior"] = -(math.log(case["vocab"]) + torch.randn(case["tokens"], generator=g, device=DEV))
    return state


# --------------------------------------------------------------------------------------- pass
def run(state):
    kind = state["kind"]
    if kind == "next":
        return dsv41_rocm.sample_next(state["logits"], state["temperature"], generator=state["generator"])
    if kind == "sample":
        r = dsv41_rocm.sample(state["logits"], uniforms=None if state["greedy"] else state["uniforms"],
                                       history=state["history"], greedy=state["greedy"], **state["knobs"])
        return {"ids": r.ids, "logprobs": r.logprobs, "kept": r.kept, "status": r.status}
    if kind == "replay":
        return dsv41_rocm.replay_log_probs(state["logits"], state["ids"], history=state["history"],
                                                    **state["knobs"])
    if kind == "loss":
        current = state["current"]
        parts = list(current.split(state["lengths"]))
        if state["loss"] == "tis":
            loss, metrics = dsv41_rocm.decoupled_token_tis_loss(parts, state["old"], state["behavior"],
                                                                    state["advantages"])
        elif state["loss"] == "grpo":
            loss, metrics = dsv41_rocm.grpo_loss(parts, state["behavior"], state["advantages"])
        else:
            loss, metrics = dsv41_rocm.grpo_loss(parts, state["behavior"], state["advantages"],
                                                     ref_log_probs=state["reference"], kl_beta=0.04)
        (grad,) = torch.autograd.grad(loss, (current,))
        return {"loss": loss.detach(), "grad": grad, "metrics": metrics}
    if kind == "masked":
        return dsv41_rocm.token_log_probs(state["hidden"], state["weight"], state["targets"], state["mask"],
                                                  state["temperature"])
    if kind == "learn":
        x, w = state["hidden"], state["weight"]
        lp, ent, _ = dsv41_rocm.selected_log_probs(x, w, state["targets"], state["temperature"])
        inputs = (x, w) if w.requires_grad else (x,)
        return {"logprobs": lp.detach(), "entropy": ent.detach(),
                "grads": torch.autograd.grad((lp, ent), inputs, state["grads"])}
    lp, ent, ratio = dsv41_rocm.selected_log_probs(state["hidden"], state["weight"], state["targets"],
                                                           state["temperature"], behavior=state["behavior"])
    out = {"logprobs": lp, "entropy": ent}
    if ratio is not None:
        out["ratio"] = ratio
    return out


def work(case):
    """Every input read once and every output written once; the multiplications of the head."""
    kind = case["kind"]
    size = 4 if case.get("dtype") == "f32" else 2
    if kind == "next":
        return {"bytes": case["vocab"] * size + 12, "flops": 0}
    if kind in ("sample", "replay"):
        penalized = case["repetition_penalty"] != 1.0 or case["presence_penalty"] or case["frequency_penalty"]
        return {"bytes": case["rows"] * (case["vocab"] * size + (8 * case["history"] if penalized else 0) + 24),
                "flops": 0}
    if kind == "loss":
        n = sum(_lengths(case))
        vectors = 3 + (case["loss"] != "grpo")  # two or three inputs and the gradient
        return {"bytes": n * 4 * vectors, "flops": 0}
    H, V = case["hidden"], case["vocab"]
    n = case["tokens"] if kind != "masked" else 0.575 * case["batch"] * case["length"]
    once = {"bytes": 2.0 * (n + V) * H + 24.0 * n, "flops": 2.0 * n * H * V}
    if kind == "learn":
        both = 1 + case["weight_grad"]
        return {"bytes": once["bytes"] + 2.0 * n * H + (2.0 * V * H if case["weight_grad"] else 0),
                "flops": (1 + both) * once["flops"]}
    return once


def tolerance(case):
    kind = case["kind"]
    if kind in ("next", "sample", "replay"):
        # ids and kept sets are exact; the log-prob is a float of a 64-bit sum, whose order may
        # change its last bit
        return {"rel": 1e-6, "max": 4e-6}
    if kind == "loss":
        return {"rel": 1e-5, "max": 1e-4}  # sums of 32-bit terms in another order
    if kind == "learn":
        return {"rel": 1e-2, "max": 0.1}  # the logit gradient and both products are rounded to bf16
    return {"rel": 2e-6, "max": 2e-5}  # 32-bit dot products and sums in another order


# -------------------------------------------------------------------------------- in 64 bits
def _processed(x, history, case):
    """z of the rows x [r, V] (64 bits), penalties over the history first."""
    if history is not None:
        count = torch.zeros_like(x).scatter_add_(1, history, torch.ones_like(history, dtype=x.dtype))
        seen = count > 0
        rp = case["repetition_penalty"]
        x = torch.where(seen, torch.where(x > 0, x / rp, x * rp) - case["frequency_penalty"] * count -
                        case["presence_penalty"], x)
    return x / case["temperature"]


def _exact_rows(z, u, case):
    """ids, log-probs and kept sizes of the processed rows z for the uniforms u (None: greedy)."""
    V = z.shape[1]
    zmax = z.max(1, keepdim=True).values
    top_k, top_p, min_p = case["top_k"], case["top_p"], case["min_p"]
    keep = torch.ones_like(z, dtype=torch.bool)
    if min_p > 0:
        keep &= z - zmax >= math.log(min_p)
    if 0 < top_k < V or top_p < 1:
        k = min(V, top_k) if 0 < top_k < V else V
        order = torch.where(keep, z, -math.inf).sort(dim=1, descending=True, stable=True)
        p = (order.values[:, :k] - zmax).exp()
        n = torch.full((z.shape[0],), k, device=z.device)
        if top_p < 1:
            cum = p.cumsum(1)
            n = (cum < top_p * cum[:, -1:]).sum(1) + 1
        chosen = torch.zeros_like(keep)
        chosen.scatter_(1, order.indices[:, :k], torch.arange(k, device=z.device)[None, :] < n[:, None])
        keep &= chosen
    p = torch.where(keep, (z - zmax).exp(), 0.0)
    total = p.sum(1)
    if u is None:
        ids = z.argmax(1)
    else:
        ids = (p.cumsum(1) <= (u.double() * total)[:, None]).sum(1).clamp_(max=V - 1)
    lp = (z.gather(1, ids[:, None]) - zmax)[:, 0] - total.log()
    return ids, lp, keep.sum(1)


def _exact_head(state, grads=None, block=8192):
    """Log-probs and entropies (and, with grads, the gradients) of scoring, the head in blocks."""
    x, w, T = state["hidden"].detach(), state["weight"].detach(), state["temperature"]
    if state["kind"] == "masked":
        x = x[state["mask"]]
        t = state["targets"][state["mask"]]
    else:
        t = state["targets"]
    V, x = w.shape[0], x.double()
    spans = [(b, min(V, b + block)) for b in range(0, V, block)]
    m = torch.full((x.shape[0],), -math.inf, dtype=torch.float64, device=x.device)
    s, a, zt = torch.zeros_like(m), torch.zeros_like(m), torch.zeros_like(m)
    for b, e in spans:
        z = x @ w[b:e].double().t() / T
        new = torch.maximum(m, z.max(1).values)
        c, p = (m - new).exp(), (z - new[:, None]).exp()
        s, a, m = s * c + p.sum(1), a * c + (p * z).sum(1), new
        inside = (t >= b) & (t < e)
        zt = torch.where(inside, z.gather(1, (t - b).clamp(0, e - b - 1)[:, None])[:, 0], zt)
    lse = m + s.log()
    lp, ent = zt - lse, lse - a / s
    if grads is None:
        return lp, ent
    g_lp, g_ent = (v.double()[:, None] for v in grads)
    dx, dw = torch.zeros_like(x), []
    for b, e in spans:
        wb = w[b:e].double()
        z = x @ wb.t() / T
        p = (z - lse[:, None]).exp()
        d = -g_lp * p + g_ent * p * ((lse - ent)[:, None] - z)
        inside = (t >= b) & (t < e)
        d[inside, t[inside] - b] += g_lp[inside, 0]
        d /= T
        dx += d @ wb
        if state["weight"].requires_grad:
            dw.append(d.t() @ x)
    return lp, ent, dx, torch.cat(dw) if dw else None


def _exact_loss(state):
    cur, adv = state["current"].detach().double().requires_grad_(), state["advantages"].double().to(DEV)
    beh = torch.cat(state["behavior"]).double()
    lengths = torch.tensor(state["lengths"], device=DEV)
    R, n = len(lengths), int(lengths.sum())
    of = torch.repeat_interleave(torch.arange(R, device=DEV), lengths)

    def mean(v):  # over the responses, of each response's mean
        return (torch.zeros(R, dtype=torch.float64, device=DEV).index_add(0, of, v) / lengths).mean()

    A = adv[of]
    old = torch.cat(state["old"]).double() if state["loss"] == "tis" else beh
    ratio = (cur - old).exp()
    s = torch.minimum(ratio * A, ratio.clamp(0.8, 1.2) * A)
    if state["loss"] == "tis":
        raw = (old - beh).exp()
        weight = raw.clamp(max=2.0)
        loss = -mean(weight * s)
        wsum, wsq, rsum, dropped = weight.sum(), (weight * weight).sum(), raw.sum(), (raw - weight).sum()
        clipped, ess = (raw > 2.0).double().sum(), wsum * wsum / wsq
        m = {"loss": loss, "policy_loss": loss, "response_count": float(R), "token_count": float(n), "is_cap": 2.0,
             "is_weight_sum": wsum, "is_weight_square_sum": wsq, "is_weight_mean": wsum / n,
             "is_weight_min": weight.min(), "is_weight_max": weight.max(), "is_raw_weight_sum": rsum,
             "is_raw_weight_min": raw.min(), "is_raw_weight_max": raw.max(), "is_clipped_tokens": clipped,
             "is_clipped_fraction": clipped / n, "is_dropped_weight_mass": dropped,
             "is_dropped_weight_mass_fraction": dropped / rsum, "is_token_weight_ess": ess,
             "is_token_weight_ess_fraction": ess / n, "native_old_minus_behavior_mean": (old - beh).mean(),
             "native_old_minus_behavior_max_abs": (old - beh).abs().max(), "native_ppo_ratio_mean": ratio.mean(),
             "native_ppo_clip_fraction": ((ratio - 1).abs() > 0.2).double().mean()}
    else:
        policy, kl = -mean(s), torch.zeros((), dtype=torch.float64, device=DEV)
        if state["loss"] == "grpo_kl":
            d = torch.cat(state["reference"]).double() - cur
            kl = mean(ratio * (torch.expm1(d) - d))
        loss = policy + 0.04 * kl
        m = {"loss": loss, "policy_loss": policy, "kl": kl, "clip_fraction": mean(((ratio - 1).abs() > 0.2).double()),
             "importance_ratio": mean(ratio), "approx_kl": mean(beh - cur)}
    (grad,) = torch.autograd.grad(loss, (cur,))
    return {"loss": loss.detach(), "grad": grad, "metrics": {k: float(v) for k, v in m.items()}}


def exact(case, seed):
    state, kind = prepare(case, seed), case["kind"]
    if kind == "next":
        u = torch.rand(1, generator=state["generator"], dtype=torch.float32).to(DEV)
        ids, lp, _ = _exact_rows(state["logits"].double() / case["temperature"], u, NO_KNOBS)
        return int(ids), float(lp)
    if kind in ("sample", "replay"):
        parts = []
        for r in range(0, case["rows"], 64):
            at = slice(r, min(case["rows"], r + 64))
            history = state["history"][at] if state["history"] is not None else None
            z = _processed(state["logits"][at].double(), history, case)
            if kind == "replay":
                parts.append((z.log_softmax(1).gather(1, state["ids"][at, None])[:, 0],))
            else:
                parts.append(_exact_rows(z, None if case["greedy"] else state["uniforms"][at], case))
        got = [torch.cat(p) for p in zip(*parts)]
        return got[0] if kind == "replay" else {"ids": got[0], "logprobs": got[1], "kept": got[2].int(), "status": None}
    if kind == "loss":
        return _exact_loss(state)
    if kind == "learn":
        lp, ent, dx, dw = _exact_head(state, state["grads"])
        return {"logprobs": lp, "entropy": ent, "grads": (dx, dw) if dw is not None else (dx,)}
    lp, ent = _exact_head(state)
    if kind == "masked":
        return torch.zeros(state["mask"].shape, dtype=lp.dtype, device=DEV).masked_scatter(state["mask"], lp)
    out = {"logprobs": lp, "entropy": ent}
    if state["behavior"] is not None:
        out["ratio"] = (lp - state["behavior"].double()).exp().clamp(max=2.0)
    return out
