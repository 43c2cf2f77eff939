"""The work whose speed is measured: one MoE layer, one expert-parallel rank's
part of a layer, and whole model steps, through the entry points that a
program calls (HipMoEBackend, HipEPShareBackend, build_hip_model).

Shapes are GraniteMoE's (hidden 1024, 32 experts, top-8, intermediate 512) as
in the tests and the benchmark, with one wider shape and one narrower one.
Sizes run from one token (decode of one sequence) to 16384 tokens (the
benchmark's skewed batch).  Inputs are made on the GPU from the seed alone:
N(0, 1) hidden states, N(0, 0.02) weights, and for skewed routing a bias
-skew * log(rank) on the router logits put into the hidden states (the router
has no bias of its own).
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(1, os.path.join(os.getcwd(), "mini-ep_amd"))

from miniep_amd import (EPStats, HipEPShareBackend, HipMoEBackend, Placement, ops, route)  # noqa: E402
from miniep_amd import model as M  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
GRANITE = dict(hidden=1024, inter=512, experts=32, top_k=8)
WORLD, RANK = 4, 1


def listed():
    return [
        # one sequence decoding: the smallest call, eight of the 32 experts' weights
        dict(name="decode_1", kind="layer", tokens=1, dtype="bf16", skew=0.0, valid=1.0, **GRANITE),
        # a decode batch: every expert's weights are read for a few rows each
        dict(name="decode_32", kind="layer", tokens=32, dtype="bf16", skew=0.0, valid=1.0, **GRANITE),
        # a larger decode batch with padded slots masked out
        dict(name="decode_100_masked", kind="layer", tokens=100, dtype="bf16", skew=0.0, valid=0.9, **GRANITE),
        # one prompt, or a chunk of one: an ordinary prefill, an odd number of tokens
        dict(name="prefill_517", kind="layer", tokens=517, dtype="bf16", skew=0.6, valid=1.0, **GRANITE),
        # eight prompts of 512 tokens in one batch
        dict(name="prefill_4096", kind="layer", tokens=4096, dtype="bf16", skew=0.6, valid=1.0, **GRANITE),
        # the benchmark's layer: hot experts get up to four times the mean load
        dict(name="skewed_16384", kind="layer", tokens=16384, dtype="bf16", skew=1.2, valid=1.0, **GRANITE),
        # the fp32 model's layer, router and backend called one after the other
        dict(name="fp32_512", kind="protocol", tokens=512, dtype="fp32", skew=0.0, valid=1.0, **GRANITE),
        # a wider model: twice the hidden and intermediate sizes, 64 experts, padded tokens
        dict(name="wide_1000", kind="protocol", tokens=1000, dtype="bf16", skew=0.6, valid=0.95, hidden=2048,
             inter=1024, experts=64, top_k=8),
        # expert parallelism, receive side: one of four ranks' share of a batch
        # from four senders, hot experts replicated
        dict(name="ep_share_8192", kind="share", tokens=8192, dtype="bf16", skew=1.1, valid=1.0, **GRANITE),
        # expert parallelism, one rank's whole step for its own tokens: send
        # buffer, experts on what arrived, combine of what came back
        dict(name="ep_step_1024", kind="ep_step", tokens=1024, dtype="bf16", skew=1.1, valid=1.0, **GRANITE),
        # the 24-layer model: one decode step of eight sequences, 512 positions cached
        dict(name="model_decode_8x512", kind="model_decode", batch=8, length=512, layers=24, dtype="bf16"),
        # the 24-layer model: eight prompts of 256 tokens, logits of the last positions
        dict(name="model_prefill_8x256", kind="model_prefill", batch=8, length=256, layers=24, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds."""
    kind = rng.choice(["layer"] * 6 + ["protocol"] * 3 + ["share"] * 2 + ["ep_step"] * 2 + ["model_decode", "model_prefill"])
    skew = rng.choice([0.0, 0.3, 0.6, 0.9, 1.2])
    valid = rng.choice([1.0, 1.0, 0.97, 0.8])
    if kind == "layer":
        return dict(kind=kind, tokens=_log(rng, 1, 16384), dtype="bf16", skew=skew, valid=valid, **GRANITE)
    if kind == "protocol":
        shape = rng.choice([GRANITE, GRANITE, dict(hidden=2048, inter=1024, experts=64, top_k=8),
                            dict(hidden=512, inter=256, experts=16, top_k=4)])
        dtype = rng.choice(["fp32", "bf16"])
        most = 16384 if dtype == "bf16" and shape["hidden"] < 2048 else 1500
        return dict(kind=kind, tokens=_log(rng, 1, most), dtype=dtype, skew=skew, valid=valid, **shape)
    if kind == "share":
        return dict(kind=kind, tokens=_log(rng, 64, 16384), dtype="bf16", skew=skew, valid=valid, **GRANITE)
    if kind == "ep_step":
        return dict(kind=kind, tokens=_log(rng, 4, 4096), dtype="bf16", skew=skew, valid=valid, **GRANITE)
    if kind == "model_decode":
        return dict(kind=kind, batch=rng.randint(1, 32), length=_log(rng, 16, 1024), layers=24, dtype="bf16")
    batch = rng.randint(1, 8)
    return dict(kind=kind, batch=batch, length=_log(rng, 16, 2048 // batch), layers=24, dtype="bf16")


# ---- inputs ------------------------------------------------------------------

def _rank_bias(experts, skew, gen, dev):
    """-skew * log(rank of the expert) under a random order of the experts, mean 0."""
    rank = torch.empty(experts, dtype=torch.float64, device=dev)
    rank[torch.randperm(experts, generator=gen, device=dev)] = torch.arange(1, experts + 1, dtype=torch.float64,
                                                                            device=dev)
    b = -skew * rank.log()
    return b - b.mean()


def _layer_inputs(case, seed):
    """x, router weights, expert weights and valid mask of one layer."""
    dev = torch.device("cuda")
    gen = torch.Generator(dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    n, h, i, e = case["tokens"], case["hidden"], case["inter"], case["experts"]
    w_r = torch.randn(e, h, generator=gen, device=dev) * 0.02
    x = torch.randn(n, h, generator=gen, device=dev)
    if case["skew"] > 0:
        b = _rank_bias(e, case["skew"], gen, dev)
        wd = w_r.double()
        x += (wd.T @ torch.linalg.solve(wd @ wd.T, b)).float()
    w_in = (torch.randn(e, 2 * i, h, generator=gen, device=dev) * 0.02).to(dt)
    w_out = (torch.randn(e, h, i, generator=gen, device=dev) * 0.02).to(dt)
    valid = torch.rand(n, generator=gen, device=dev) < case["valid"] if case["valid"] < 1.0 else None
    return x.to(dt), w_r.to(dt), w_in, w_out, valid


def _owners(case):
    """One layer's placement over four ranks: contiguous blocks of experts, and
    a second and third copy of some experts, as the balancer gives hot ones."""
    gen = torch.Generator().manual_seed(2)
    e, per = case["experts"], case["experts"] // WORLD
    owners = [[j // per] for j in range(e)]
    for c, j in enumerate(torch.randperm(e, generator=gen)[: e // 4].tolist()):
        more = [(owners[j][0] + 1 + c) % WORLD, (owners[j][0] + 3) % WORLD][: 1 + c % 2]
        owners[j] = sorted(set(owners[j] + more))
    return owners


def _topk_softmax(logits, k):
    v, idx = logits.topk(k, dim=-1)
    return idx, torch.softmax(v, -1)


def _model_config(case):
    return M.ModelConfig(num_hidden_layers=case["layers"])


def _model_weights(case, seed):
    """Random weights under the checkpoint's names, N(0, 0.02), drawn on the GPU."""
    cfg = _model_config(case)
    dev = torch.device("cuda")
    gen = torch.Generator(dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    h, i, e = cfg.hidden_size, cfg.intermediate_size, cfg.num_local_experts
    q, kv = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim

    def mat(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=dt) * 0.02

    w = {"model.embed_tokens.weight": mat(cfg.vocab_size, h), "model.norm.weight": torch.ones(h, dtype=dt, device=dev)}
    for layer in range(cfg.num_hidden_layers):
        p = f"model.layers.{layer}."
        w[p + "input_layernorm.weight"] = torch.ones(h, dtype=dt, device=dev)
        w[p + "post_attention_layernorm.weight"] = torch.ones(h, dtype=dt, device=dev)
        w[p + "self_attn.q_proj.weight"] = mat(q, h)
        w[p + "self_attn.k_proj.weight"] = mat(kv, h)
        w[p + "self_attn.v_proj.weight"] = mat(kv, h)
        w[p + "self_attn.o_proj.weight"] = mat(h, q)
        w[p + "block_sparse_moe.router.layer.weight"] = mat(e, h)
        w[p + "block_sparse_moe.input_linear.weight"] = mat(e, 2 * i, h)
        w[p + "block_sparse_moe.output_linear.weight"] = mat(e, h, i)
    ids = torch.randint(0, cfg.vocab_size, (case["batch"], case["length"] + 1), generator=gen, device=dev)
    return cfg, w, ids


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("layer", "protocol"):
        x, w_r, w_in, w_out, valid = _layer_inputs(case, seed)
        return dict(kind=kind, x=x, w_r=w_r, valid=valid, k=case["top_k"], backend=HipMoEBackend(w_in, w_out))
    if kind in ("share", "ep_step"):
        x, w_r, w_in, w_out, valid = _layer_inputs(case, seed)
        k, n = case["top_k"], case["tokens"]
        placement = Placement([_owners(case)])
        mine = placement.experts_of_rank(RANK)[0]
        stats = EPStats(1, case["experts"])
        be = HipEPShareBackend(0, placement, RANK, w_in[mine], w_out[mine], stats=stats, check=False)
        # the router's results, from 64-bit logits: a near-tie then falls the same way in exact()
        idx, gate = _topk_softmax(x.double() @ w_r.double().T, k)
        s = dict(kind=kind, x=x, idx=idx, gate=gate.to(x.dtype), valid=valid, backend=be)
        if kind == "share":
            s["segments"] = [n * r // WORLD for r in range(WORLD + 1)]
            s["y"] = torch.zeros(n * k, case["hidden"], dtype=x.dtype, device=x.device)
        else:
            s["recv_x"], s["recv_experts"], s["back"] = _arrived(case, seed, x, mine)
        return s
    cfg, w, ids = _model_weights(case, seed)
    model = M.build_hip_model(cfg, w)
    prompt = ids[:, : case["length"]]
    last = torch.full((case["batch"],), case["length"] - 1, device=ids.device)
    if kind == "model_prefill":
        return dict(kind=kind, model=model, cfg=cfg, prompt=prompt, last=last, room=case["length"] + 32)
    cache = M.KVCache(cfg, case["batch"], case["length"] + 32, ids.device)
    model(prompt, cache=cache, logits_at=last)
    return dict(kind=kind, model=model, cache=cache, length=case["length"], token=ids[:, case["length"]:])


def _arrived(case, seed, x, mine):
    """What the two all-to-alls bring a rank: rows for its own experts (as
    many as it sends on average), and the expert outputs of its own rows."""
    gen = torch.Generator(x.device).manual_seed(seed + 1)
    rows = case["tokens"] * case["top_k"]
    recv_x = torch.randn(rows, case["hidden"], generator=gen, device=x.device).to(x.dtype)
    pick = torch.randint(0, len(mine), (rows,), generator=gen, device=x.device)
    recv_experts = torch.tensor(mine, device=x.device)[pick]
    back = (torch.randn(rows, case["hidden"], generator=gen, device=x.device) * 0.1).to(x.dtype)
    return recv_x, recv_experts, back


def run(s):
    kind = s["kind"]
    if kind == "layer":
        out, idx, gate = s["backend"].route_and_call(s["x"], s["w_r"], s["k"], s["valid"])
        return {"out": out, "idx": idx, "gate": gate}
    if kind == "protocol":
        idx, gate = route(s["x"], s["w_r"], s["k"])
        return {"out": s["backend"](s["x"], idx, gate, s["valid"]), "idx": idx, "gate": gate}
    if kind == "share":
        disp, y = s["backend"].share(s["x"], s["idx"], s["valid"], s["segments"], y_entries=s["y"])
        return {"y": y, "counts": disp.counts, "row_of_entry": disp.row_of_entry}
    if kind == "ep_step":
        sent = s["backend"].send(s["x"], s["idx"], s["valid"])
        y = s["backend"].receive(s["recv_x"], s["recv_experts"])
        out = ops.combine_rows(s["back"], s["gate"], sent.inv, s["valid"])
        return {"send_x": sent.x, "send_experts": sent.experts, "send_counts": sent.send_counts, "y": y, "out": out}
    if kind == "model_prefill":
        cache = M.KVCache(s["cfg"], s["prompt"].shape[0], s["room"], s["prompt"].device)
        return s["model"](s["prompt"], cache=cache, logits_at=s["last"])
    s["cache"].length = s["length"]          # the position that this step fills
    return s["model"](s["token"], cache=s["cache"])


# ---- the work of one pass --------------------------------------------------------

def _experts_work(rows, tokens, hidden, inter, experts, k, size):
    """(bytes of the expert weights that `tokens` tokens touch, flops of `rows` rows)."""
    touched = experts * (1.0 - (1.0 - k / experts) ** tokens)
    return touched * 3 * hidden * inter * size, 6.0 * rows * hidden * inter


def work(case):
    kind = case["kind"]
    if kind.startswith("model"):
        cfg = _model_config(case)
        b, length, h, size = case["batch"], case["length"], cfg.hidden_size, 2
        q, kv = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
        n = b if kind == "model_decode" else b * length
        wb, wf = _experts_work(n * 8, n, h, cfg.intermediate_size, cfg.num_local_experts, 8, size)
        proj = h * (2 * q + 2 * kv)
        keys = length + 1 if kind == "model_decode" else (length + 1) / 2      # causal: half the positions on average
        cached = 2 * 4 * kv * (b * (length + 1) if kind == "model_decode" else n)  # fp32 keys and values
        per = dict(bytes=wb + proj * size + cached, flops=wf + 2.0 * n * proj + 4.0 * n * keys * q)
        return {"bytes": cfg.num_hidden_layers * per["bytes"] + size * cfg.vocab_size * h + 4.0 * b * cfg.vocab_size,
                "flops": cfg.num_hidden_layers * per["flops"] + 2.0 * b * cfg.vocab_size * h}
    n, h, i, e, k = (case[f] for f in ("tokens", "hidden", "inter", "experts", "top_k"))
    size = 2 if case["dtype"] == "bf16" else 4
    live = n * case["valid"]
    if kind in ("layer", "protocol"):
        wb, wf = _experts_work(live * k, live, h, i, e, k, size)
        return {"bytes": wb + 2 * n * h * size + e * h * size + n * k * (8 + size), "flops": wf + 2.0 * n * h * e}
    if kind == "share":
        rows = live * k / WORLD
        wb, wf = _experts_work(rows, live, h, i, 1.25 * e / WORLD, min(k, 1.25 * e / WORLD), size)
        return {"bytes": wb + n * h * size + rows * h * size + n * k * (8 + 4), "flops": wf}
    rows = n * k
    sent = live * k
    wb, wf = _experts_work(rows, rows, h, i, 1.25 * e / WORLD, 1.0, size)
    send = n * h * size + sent * h * size + n * k * 8 + sent * 8
    receive = wb + 2 * rows * h * size + rows * 8
    combine = sent * h * size + n * h * size + n * k * (4 + size)
    return {"bytes": send + receive + combine, "flops": wf}


def tolerance(case):
    if case["dtype"] == "fp32":
        # sums of 512 and 1024 products in fp32; near-ties of the router may swap two slots
        return {"rel": 1e-5, "differ": 1e-4}
    if case["kind"].startswith("model"):
        # 24 layers in bf16: a changed rounding in one travels through the rest
        # (the logits are 1.3e-2 to 1.8e-2 off those in 64 bits)
        return {"rel": 3e-2}
    # activations and expert outputs rounded to bf16 once each, another order of sums
    return {"rel": 8e-3, "differ": 1e-4}


# ---- the same in 64 bits ------------------------------------------------------------

def _experts64(x, expert_of_row, w_in, w_out):
    """Output of expert expert_of_row[r] (< 0: zero) for every row of x, in fp64."""
    out = torch.zeros(x.shape[0], x.shape[1], dtype=torch.float64, device=x.device)
    inter = w_out.shape[2]
    for e in range(w_in.shape[0]):
        rows = (expert_of_row == e).nonzero().flatten()
        for r in rows.split(16384):
            h = x[r].double() @ w_in[e].double().T
            out[r] = (F.silu(h[:, :inter]) * h[:, inter:]) @ w_out[e].double().T
    return out


def _moe64(x, w_r, w_in, w_out, valid, k):
    """(layer output, gates) in fp64; experts run slot by slot to bound the memory."""
    xd = x.double()
    v, idx = (xd @ w_r.double().T).topk(k, dim=-1)
    gate = torch.softmax(v, -1)
    out = torch.zeros_like(xd)
    for s in range(k):
        e = idx[:, s] if valid is None else torch.where(valid, idx[:, s], -1)
        out += gate[:, s:s + 1] * _experts64(x, e, w_in, w_out)
    return out, gate


def _destinations(idx, valid, owners, segments):
    """Destination rank of every (token, slot) entry, -1 for masked tokens: the
    w-th entry of an expert within a sender's tokens goes to owner w mod R."""
    flat = idx.reshape(-1).tolist()
    k = idx.shape[1]
    live = [True] * idx.shape[0] if valid is None else valid.tolist()
    dest = []
    for lo, hi in zip(segments, segments[1:]):
        seen = [0] * len(owners)
        for f in range(lo * k, hi * k):
            e = flat[f]
            if not live[f // k]:
                dest.append(-1)
                continue
            dest.append(owners[e][seen[e] % len(owners[e])])
            seen[e] += 1
    return torch.tensor(dest, device=idx.device)


def _model64(cfg, w, ids):
    """Logits of the last position, in fp64, one sequence's attention at a time."""
    b, t = ids.shape
    d, hq, hk = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    dev = ids.device
    inv = cfg.rope_theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=dev) / d)
    ang = torch.arange(t, dtype=torch.float64, device=dev)[:, None] * inv[None]
    cos, sin = torch.cat([ang, ang], -1).cos(), torch.cat([ang, ang], -1).sin()

    def norm(z, weight):
        return weight.double() * z * torch.rsqrt(z.pow(2).mean(-1, keepdim=True) + cfg.rms_norm_eps)

    def rotate(z):
        return z * cos + torch.cat([-z[..., d // 2:], z[..., : d // 2]], -1) * sin

    mask = torch.full((t, t), -math.inf, dtype=torch.float64, device=dev).triu(1)
    h = w["model.embed_tokens.weight"][ids].double() * cfg.embedding_multiplier
    for layer in range(cfg.num_hidden_layers):
        p = f"model.layers.{layer}."
        x = norm(h, w[p + "input_layernorm.weight"])
        att = []
        for s in range(b):
            q, k, v = ((x[s] @ w[p + f"self_attn.{m}_proj.weight"].double().T).view(t, -1, d).transpose(0, 1)
                       for m in ("q", "k", "v"))
            q, k = rotate(q), rotate(k)
            k, v = (z.repeat_interleave(hq // hk, 0) for z in (k, v))
            a = torch.softmax(q @ k.transpose(1, 2).contiguous() * cfg.attention_multiplier + mask, -1) @ v
            att.append(a.transpose(0, 1).reshape(t, hq * d) @ w[p + "self_attn.o_proj.weight"].double().T)
        h = h + torch.stack(att) * cfg.residual_multiplier
        x = norm(h, w[p + "post_attention_layernorm.weight"]).view(b * t, -1)
        m = p + "block_sparse_moe."
        out, _ = _moe64(x, w[m + "router.layer.weight"], w[m + "input_linear.weight"], w[m + "output_linear.weight"],
                        None, cfg.num_experts_per_tok)
        h = h + out.view(b, t, -1) * cfg.residual_multiplier
    x = norm(h[:, -1:], w["model.norm.weight"])
    return x @ w["model.embed_tokens.weight"].double().T / cfg.logits_scaling


def exact(case, seed):
    kind = case["kind"]
    if kind in ("layer", "protocol"):
        x, w_r, w_in, w_out, valid = _layer_inputs(case, seed)
        out, gate = _moe64(x, w_r, w_in, w_out, valid, case["top_k"])
        return {"out": out, "idx": None, "gate": gate}
    if kind in ("share", "ep_step"):
        x, w_r, w_in, w_out, valid = _layer_inputs(case, seed)
        k, n = case["top_k"], case["tokens"]
        idx, gate = _topk_softmax(x.double() @ w_r.double().T, k)
        owners = _owners(case)
        mine = [e for e in range(case["experts"]) if RANK in owners[e]]
        if kind == "share":
            dest = _destinations(idx, valid, owners, [n * r // WORLD for r in range(WORLD + 1)])
            e = torch.where(dest == RANK, idx.reshape(-1), -1)
            y = torch.cat([_experts64(xs.repeat_interleave(k, 0), es, w_in, w_out)
                           for xs, es in zip(x.split(4096), e.split(4096 * k))])
            return {"y": y, "counts": None, "row_of_entry": None}
        dest = _destinations(idx, valid, owners, [0, n])
        order = torch.argsort(torch.where(dest < 0, WORLD, dest), stable=True)[: int((dest >= 0).sum())]
        inv = torch.full((n * k,), -1, device=x.device)
        inv[order] = torch.arange(order.numel(), device=x.device)
        recv_x, recv_experts, back = _arrived(case, seed, x, mine)
        rows = back.double()[inv.clamp(min=0)] * (inv >= 0).double()[:, None]
        return {"send_x": x[order // k].double(), "send_experts": None, "send_counts": None,
                "y": _experts64(recv_x, recv_experts, w_in, w_out),
                "out": (rows.view(n, k, -1) * gate.double()[..., None]).sum(1)}
    cfg, w, ids = _model_weights(case, seed)
    return _model64(cfg, w, ids if kind == "model_decode" else ids[:, : case["length"]])
