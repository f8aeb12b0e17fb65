"""The work this engine is measured by: steps of served models, as a program that drives the
``ModelRunner`` has them run.

A case is a model (a preset or one of the benchmark's layer sizes, random weights) and one of

* ``prompt``: whole prompts read in one step, the logits of their last tokens;
* ``mixed``: a step of chunked prefill: portions of prompts that are cached so far, beside single
  decoded tokens of other requests;
* ``decode``: one step behind cached contexts whose logits are asked for, then decode steps through the
  captured path (``decode_run``);
* ``reply``: short prompts read and then decoded behind, for models with per-request state (their
  state begins anew with each prompt, so a pass can be repeated).

Decode steps are ``runs`` calls of ``decode_run`` of ``steps`` steps.  With ``steps`` above one the device
feeds the tokens back itself; otherwise the tokens of every step are given, as in a replayed trace.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

import kvforge_amd
from kvforge_amd import ModelRunner, SamplingParams, StepEntry, Transformer
from kvforge_amd.config.presets import depolix_stack, rudorax_stack

BLOCK = 16              # tokens of a cache page, the engine's default
PORTION = 2048          # tokens a step may bring, the engine's default
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}

# the layer sizes that bench.py measures the two designs at
RUDORAX = {"w1024": dict(vocab=32000, width=1024, pairs=4, heads=16, kv_heads=4, dim=64, window=1024, lstm_heads=4,
                         lstm_dim=128, lstm_vdim=256, ff=512, experts=16, top=2, identity=2, shared_ff=1024),
           "w2048": dict(vocab=128256, width=2048, pairs=4, heads=32, kv_heads=8, dim=64, window=1024, lstm_heads=8,
                         lstm_dim=128, lstm_vdim=256, ff=1024, experts=32, top=4, identity=2, shared_ff=2048)}
DEPOLIX = {"w1024": dict(vocab=32000, width=1024, groups=2, heads=16, latent_dim=64, rot_dim=32, q_rank=384, kv_rank=192,
                         att_heads=16, att_kv_heads=4, att_dim=64, window=1024, mem_heads=8, mem_kv_heads=4, mem_dim=128,
                         mem_vdim=128, gate_rank=128, ff=4096, moe_ff=1024, experts=16, top=4),
           "w2048": dict(vocab=128256, width=2048, groups=2, heads=32, latent_dim=64, rot_dim=32, q_rank=768, kv_rank=192,
                         att_heads=32, att_kv_heads=8, att_dim=64, window=1024, mem_heads=16, mem_kv_heads=8, mem_dim=128,
                         mem_vdim=128, gate_rank=128, ff=8192, moe_ff=2048, experts=32, top=4)}


# ------------------------------------------------------------------------------------- cases
def _case(model, kind, prompts, singles=(), dtype="bfloat16", layers=0, runs=0, steps=0, sampled=False):
    """``prompts``: ``tokens@cached`` of every run of tokens, ``singles``: cached tokens of every request
    that decodes, both as texts.  ``layers``: the model is cut to so many (0: all of them)."""
    return {"model": model, "kind": kind, "dtype": dtype, "layers": layers, "runs": runs, "steps": steps,
            "sampled": sampled, "prompts": " ".join(f"{n}@{c}" for n, c in prompts),
            "singles": " ".join(str(c) for c in singles)}


def listed():
    rng = random.Random(7)
    return [dict(c, name=n) for n, c in (
        # a small model answering one user: the latency of a step
        ("small_decode_b1", _case("small", "decode", (), (57,), runs=1, steps=8)),
        # the served default: a batch of eight chats, the device taking eight steps by itself
        ("llama1b_decode_b8", _case("llama-1b", "decode", (), [rng.randint(520, 700) for _ in range(8)], runs=1, steps=8)),
        # a loaded server: many requests at uneven depths, drawn with temperature and top-p
        ("llama1b_decode_b41_sampled", _case("llama-1b", "decode", (), [rng.randint(60, 2900) for _ in range(41)],
                                             runs=8, steps=1, sampled=True)),
        # long documents behind wide heads (some layers of the 8B shape)
        ("llama8b_decode_long", _case("llama-8b", "decode", (), (12011, 16200, 9001, 14333), layers=4, runs=8, steps=1)),
        # time to the first token: a short question, and a prompt that fills a step
        ("llama1b_prompt_61", _case("llama-1b", "prompt", [(61, 0)])),
        ("llama1b_prompt_2048", _case("llama-1b", "prompt", [(2048, 0)])),
        # a step of chunked prefill: a late portion, an early one and a fresh prompt beside decodes
        ("llama1b_mixed", _case("llama-1b", "mixed", [(1013, 3072), (511, 512), (333, 0)],
                                [rng.randint(100, 1800) for _ in range(19)])),
        # the 32-bit engine, its default type: checking a model against another implementation
        ("llama1b_prompt_fp32", _case("llama-1b", "prompt", [(777, 0)], dtype="float32")),
        # window attention with a sink, matrix memories, routed experts: prompts, and a reply
        ("rudorax_prompts", _case("rudorax-w2048", "prompt", [(1301, 0), (741, 0)])),
        ("rudorax_reply_b8", _case("rudorax-w2048", "reply", [(rng.randint(16, 60), 0) for _ in range(8)], runs=8, steps=1)),
        # latent attention, window attention beside a delta-rule memory, experts: a long prompt, and a reply
        ("depolix_prompt", _case("depolix-w2048", "prompt", [(2047, 0)])),
        ("depolix_reply_b5", _case("depolix-w2048", "reply", [(rng.randint(16, 60), 0) for _ in range(5)], runs=8, steps=1)),
    )]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cut(rng, total, most):
    """``total`` tokens as one to ``most`` ragged runs of at least two tokens."""
    parts = rng.randint(1, max(1, min(most, total // 16)))
    at = sorted(rng.sample(range(2, total - 1, 2), parts - 1)) if parts > 1 else []
    return [b - a for a, b in zip([0] + at, at + [total])]


def draw(rng):
    family = rng.choice(["llama", "llama", "llama", "rudorax", "depolix"])
    if family != "llama":
        model = f"{family}-{rng.choice(['w1024', 'w2048'])}"
        if rng.random() < 0.6:
            return _case(model, "prompt", [(n, 0) for n in _cut(rng, _log_int(rng, 40, PORTION), 6)])
        return _case(model, "reply", [(_log_int(rng, 5, 60), 0) for _ in range(_log_int(rng, 1, 8))], runs=8, steps=1)
    kind = rng.choice(["prompt", "mixed", "decode", "decode"])
    if kind == "prompt":
        dtype = "float32" if rng.random() < 0.25 else "bfloat16"
        most = 777 if dtype == "float32" else PORTION
        return _case(rng.choice(["small", "llama-1b", "llama-1b"]), "prompt",
                     [(n, 0) for n in _cut(rng, _log_int(rng, 20, most), 6)], dtype=dtype)
    if kind == "mixed":
        runs = [(n, rng.choice([0, BLOCK * rng.randint(1, 128), rng.randint(1, 2048)]))
                for n in _cut(rng, _log_int(rng, 60, 1857), 3)]
        return _case("llama-1b", "mixed", runs, [_log_int(rng, 10, 1800) for _ in range(_log_int(rng, 1, 19))])
    if rng.random() < 0.2:
        return _case("llama-8b", "decode", (), [_log_int(rng, 500, 14000) for _ in range(rng.randint(1, 3))],
                     layers=4, runs=8, steps=1)
    model, sampled = rng.choice(["small", "llama-1b", "llama-1b"]), rng.random() < 0.4
    return _case(model, "decode", (), [_log_int(rng, 20, 1900) for _ in range(_log_int(rng, 1, 41))],
                 runs=8 if sampled else 1, steps=1 if sampled else 8, sampled=sampled)


def _sizes(case):
    """(tokens, cached tokens before them) of every run, cached tokens of every single."""
    runs = [tuple(int(x) for x in t.split("@")) for t in case["prompts"].split()]
    return runs, [int(x) for x in case["singles"].split()]


def _config(case):
    family, _, size = case["model"].partition("-")
    if family == "rudorax":
        return rudorax_stack(**RUDORAX[size], max_positions=8192)
    if family == "depolix":
        return depolix_stack(**DEPOLIX[size], max_positions=8192)
    cfg = kvforge_amd.preset_dict(case["model"])
    if case["layers"]:
        cfg["num_hidden_layers"] = case["layers"]
    return cfg


def _vocab(case):
    cfg = _config(case)
    return cfg["vocab_size"] if "vocab_size" in cfg else cfg["vocab"]


def _drawn(case, seed):
    """The case's model with random weights, and the weights as they were drawn."""
    weights: dict[str, torch.Tensor] = {}
    model = Transformer.from_random(_config(case), seed, DTYPES[case["dtype"]], "cuda", drawn=weights)
    return model, weights


def _sequences(case, seed):
    """Token ids of every request, runs first: what is cached, what the pass brings, and behind it
    the tokens of the decode steps."""
    runs, singles = _sizes(case)
    rng = np.random.default_rng([int(seed), 20])
    more = case["runs"] * case["steps"] + 1
    return [rng.integers(1, _vocab(case), c + n + more).tolist()
            for n, c in runs + [(0, c) for c in singles]]


# ------------------------------------------------------------------------------------- the pass
def prepare(case, seed):
    """A runner with the model and its cache, the contexts read, every request's pages taken."""
    runs, singles = _sizes(case)
    seqs = _sequences(case, seed)
    counts = [(c, n) for n, c in runs] + [(c, 0) for c in singles]
    more = case["runs"] * case["steps"] + 1
    pages = sum(-(-len(s) // BLOCK) for s in seqs)
    longest = max(len(s) for s in seqs)
    runner = ModelRunner(_drawn(case, seed)[0], BLOCK, pages + 8, max_num_seqs=len(seqs),
                         max_num_batched_tokens=PORTION, max_model_len=-(-longest // 64) * 64)
    ids = [f"r{i}" for i in range(len(seqs))]
    for rid, s, (c, _) in zip(ids, seqs, counts):
        runner.cache.allocate(rid, len(s))
        for lo in range(0, c, PORTION):
            runner.step([StepEntry(rid, s[lo:min(c, lo + PORTION)], lo, "none")])
    if case["kind"] == "mixed":
        first = [StepEntry(r, s[c:c + n] if n else s[c:c + 1], c, "last") for r, s, (c, n) in zip(ids, seqs, counts)]
    else:
        first = [StepEntry(r, s[c:c + n], c, "last") for r, s, (c, n) in zip(ids, seqs, counts) if n]
    singles_at = [[StepEntry(r, s[c + n + j:c + n + j + 1], c + n + j, "last") for r, s, (c, n) in zip(ids, seqs, counts)]
                  for j in range(more)] if case["runs"] else []
    how = dict(temperature=0.8, top_p=0.9) if case["sampled"] else dict(temperature=0.0)
    torch.cuda.synchronize()
    return {"runner": runner, "first": first, "singles": singles_at, "case": case,
            "params": [SamplingParams(max_tokens=more, ignore_eos=True, **how) for _ in seqs]}


def run(state):
    runner, case = state["runner"], state["case"]
    out = {}
    if state["first"]:
        logits = runner.step(state["first"])
        if not case["runs"]:
            return {"logits": logits}
        out["prompt_logits"] = logits.clone()      # the next step writes over them
    out["logits"] = runner.step(state["singles"][0]).clone()
    b, k = len(state["params"]), case["steps"]
    tokens = []
    for j in range(1, 1 + case["runs"] * k, k):
        tokens += runner.decode_run(state["singles"][j], 0, state["params"], list(range(b)), [j] * b, k)
    out["tokens"] = np.asarray(tokens, dtype=np.int64)
    return out


# ------------------------------------------------------------------------------------- what it cannot do without
def _model_work(case):
    """(parameters every token is multiplied with, the head's among them not; the head's; parameters
    of one routed expert, how many, chosen, in how many layers; cached values a token and layer
    group: (layers, values, multiply-adds per query and key, window); state values a request, read
    and written; multiply-adds of the memories a token)."""
    family, _, size = case["model"].partition("-")
    if family == "rudorax":
        c = RUDORAX[size]
        w, p = c["width"], c["pairs"]
        attn = w * c["dim"] * 2 * (c["heads"] + c["kv_heads"])
        mem = w * (2 * c["lstm_heads"] * c["lstm_dim"] + 3 * c["lstm_heads"] * c["lstm_vdim"] + 2 * c["lstm_heads"])
        fixed = p * (attn + mem) + 2 * p * (3 * w * c["shared_ff"] + w * (c["experts"] + c["identity"]))
        cell = p * c["lstm_heads"] * c["lstm_dim"] * c["lstm_vdim"]
        return (fixed, c["vocab"] * w, (3 * w * c["ff"], c["experts"], c["top"], 2 * p),
                [(p, 2 * c["kv_heads"] * c["dim"], 2 * c["heads"] * c["dim"], c["window"])], cell, 2 * cell)
    if family == "depolix":
        c = DEPOLIX[size]
        w, n, h = c["width"], 2 * c["groups"], c["heads"]
        latent = (w * (c["q_rank"] + c["kv_rank"] + c["rot_dim"] + 2 * h * c["latent_dim"])
                  + c["q_rank"] * h * (c["latent_dim"] + c["rot_dim"]) + 2 * h * c["latent_dim"] * c["kv_rank"])
        left = w * (2 * (c["att_heads"] + c["att_kv_heads"]) * c["att_dim"] + c["att_heads"])
        right = (w * (2 * c["mem_kv_heads"] * c["mem_dim"] + 2 * c["mem_heads"] * c["mem_vdim"] + 2 * c["gate_rank"]
                      + c["mem_heads"]) + c["gate_rank"] * c["mem_heads"] * (c["mem_dim"] + c["mem_vdim"]))
        fixed = n * (latent + left + right + 3 * w * c["ff"] + w * c["experts"])
        cell = n * c["mem_heads"] * c["mem_dim"] * c["mem_vdim"]
        # a prompt's queries meet keys and values of every head: the cheaper way round
        groups = [(n, c["kv_rank"] + c["rot_dim"], h * (2 * c["latent_dim"] + c["rot_dim"]), None),
                  (n, 2 * c["att_kv_heads"] * c["att_dim"], 2 * c["att_heads"] * c["att_dim"], c["window"])]
        return fixed, c["vocab"] * w, (3 * w * c["moe_ff"], c["experts"], c["top"], n), groups, cell, 3 * cell
    c = _config(case)
    w, L = c["hidden_size"], c["num_hidden_layers"]
    d, h, kv = c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"]
    fixed = L * (w * d * 2 * (h + kv) + 3 * w * c["intermediate_size"])
    return fixed, c["vocab_size"] * w, (0, 1, 0, 0), [(L, 2 * kv * d, 2 * h * d, None)], 0, 0


def work(case):
    fixed, head, (expert, experts, top, moe_layers), groups, cell, mem_macs = _model_work(case)
    elem = 2 if case["dtype"] == "bfloat16" else 4
    vocab = _vocab(case)
    runs, singles = _sizes(case)
    forwards = []                                  # (tokens, cached) of every sequence of a forward
    if case["kind"] == "mixed":
        forwards.append(runs + [(1, c) for c in singles])
    elif runs:
        forwards.append(runs)
    ends = [n + c for n, c in runs] + singles
    for j in range(case["runs"] * case["steps"] + (1 if case["runs"] else 0)):
        forwards.append([(1, c + j) for c in ends])
    total = flops = 0.0
    for seqs in forwards:
        n = sum(t for t, _ in seqs)
        rows = len(seqs)
        touched = experts * (1.0 - (1.0 - top / experts) ** n) if moe_layers else 0.0
        total += elem * (fixed + head + moe_layers * touched * expert)
        flops += 2.0 * (n * (fixed + moe_layers * top * expert + mem_macs) + rows * head)
        for t, c in seqs:
            total += 8.0 * cell
            for layers, values, macs, window in groups:
                pairs = sum(min(c + i + 1, window) for i in range(t)) if window else t * c + t * (t + 1) / 2
                total += elem * layers * values * ((min(c, window) if window else c) + t)
                flops += 2.0 * layers * macs * pairs
        total += 4.0 * rows * vocab
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Four times what was seen.  Logits against 64 bits: in float32 1e-5; in bfloat16 0.007 for the
    small model, 0.02 to 0.03 for the others, whose attention is peaked or whose routers meet near ties
    (a routed layer that falls the other way moves a row by 0.05 to 0.1).  Tokens of given steps: one in
    sixteen stands that near a tie.  Tokens fed back differ behind the first that does; drawn ones out of
    thousands of nearly equal candidates differ with the last bits of the sums before them."""
    if case["dtype"] == "float32":
        return {"rel": 4e-5, "differ": 0.05}
    differ = 1.0 if case["sampled"] else 0.25 if case["steps"] == 1 else 0.6
    return {"rel": 0.03 if case["model"] == "small" else 0.1, "differ": differ}


# ------------------------------------------------------------------------------------- in 64 bits
def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _angles(freq, T):
    """Cosine and sine of every position's angles, which are 32-bit numbers by definition."""
    a = torch.arange(T, dtype=torch.float32, device="cuda")[:, None] * freq.to(device="cuda", dtype=torch.float32)
    return a.cos().double()[:, None], a.sin().double()[:, None]


def _turn_pairs(x, freq, mag=1.0):
    """Neighbouring elements of the first ``2 len(freq)`` of every head turned by the position's angles."""
    cos, sin = (t * mag for t in _angles(freq, x.shape[0]))
    n = 2 * len(freq)
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    return torch.cat([torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2), x[..., n:]], -1)


def _attend(q, k, v, scale, window=None, sink=None, keep=0, bias=None):
    """Causal attention of ``q [T, H, d]`` over ``k, v [T, KV, .]``, a block of queries at a time; ``bias [distance, H]``."""
    T, H = q.shape[:2]
    group = H // k.shape[1]
    kk, vv = (t.transpose(0, 1).repeat_interleave(group, 0).contiguous() for t in (k, v))
    out = []
    for lo in range(0, T, 512):
        hi = min(T, lo + 512)
        s = torch.matmul(q[lo:hi].transpose(0, 1).contiguous(), kk[:, :hi].transpose(1, 2).contiguous()) * scale
        away = torch.arange(lo, hi, device=q.device)[:, None] - torch.arange(hi, device=q.device)
        if bias is not None:
            s += bias[away.clamp(min=0)].permute(2, 0, 1)
        s.masked_fill_((away < 0) | ((away >= (window or T + 1)) & (torch.arange(hi, device=q.device) >= keep)), -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(H, hi - lo, 1)], -1)
        p = torch.softmax(s, -1)[..., :hi]
        out.append(torch.matmul(p, vv[:, :hi]).transpose(0, 1))
    return torch.cat(out)


def _llama3_frequencies(cfg):
    d, s = cfg["head_dim"], cfg.get("rope_scaling")
    freq = 1.0 / (cfg["rope_theta"] ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    if not s:
        return freq
    turns = s["original_max_position_embeddings"] * freq.double() / (2 * math.pi)
    keep = ((turns - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])).clamp(0, 1)
    return ((1 - keep) * freq.double() / s["factor"] + keep * freq.double()).float()


def _llama_rows(cfg, w, ids):
    H, KV, d, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    T = len(ids)
    cos, sin = _angles(_llama3_frequencies(cfg), T)

    def turn(x):
        u, v = x.chunk(2, -1)
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

    x = w("model.embed_tokens.weight")[ids]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        a = _rms(x, eps) * w(p + "input_layernorm.weight")
        q, k, v = ((a @ w(p + f"self_attn.{n}_proj.weight").T).view(T, -1, d) for n in "qkv")
        o = _attend(turn(q), turn(k), v, d ** -0.5)
        x = x + o.reshape(T, H * d) @ w(p + "self_attn.o_proj.weight").T
        a = _rms(x, eps) * w(p + "post_attention_layernorm.weight")
        x = x + (F.silu(a @ w(p + "mlp.gate_proj.weight").T) * (a @ w(p + "mlp.up_proj.weight").T)) @ w(p + "mlp.down_proj.weight").T
    return _rms(x, eps) * w("model.norm.weight")


def _gated(h, w, p, sep="."):
    return (F.silu(h @ w(p + sep + "gate").T) * (h @ w(p + sep + "up").T)) @ w(p + sep + "down").T


def _yarn_frequencies(rot):
    dims, base, s = rot["dims"], rot["base"], rot["scaling"]
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = base ** (-2.0 * i / dims)
    where = [dims * math.log(s["original"] / (2 * math.pi * s[n])) / (2 * math.log(base)) for n in ("fast", "slow")]
    lo, hi = max(math.floor(where[0]), 0), min(math.ceil(where[1]), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def _mlstm(h, w, p, m, eps):
    T, H, d, dv, cap = h.shape[0], m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q, k, v = ((h @ w(f"{p}.{n}").T).view(T, H, -1) for n in "qkv")
    q = q * d ** -0.5
    li, lf = (cap * torch.tanh((h @ w(f"{p}.{n}").T + w(f"{p}.{n}.b")) / cap) for n in "if")
    lf = F.logsigmoid(lf)
    S, n, top = h.new_zeros(H, d, dv), h.new_zeros(H, d), h.new_zeros(H)
    out = h.new_empty(T, H, dv)
    for t in range(T):
        a = lf[t] + top
        top = torch.maximum(a, li[t])
        keep, take = torch.exp(a - top), torch.exp(li[t] - top)[:, None] * k[t]
        S = torch.baddbmm(keep[:, None, None] * S, take[:, :, None], v[t][:, None, :])
        n = keep[:, None] * n + take
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        out[t] = torch.bmm(q[t][:, None, :], S)[:, 0] / den[:, None]
    o = _rms(out, eps).reshape(T, H * dv) * w(p + ".norm") * torch.sigmoid(h @ w(p + ".g").T)
    return o @ w(p + ".o").T


def _rudorax_rows(cfg, w, ids):
    eps, T = cfg["norm"]["eps"], len(ids)
    x = w("embed")[ids] * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        p, m, r = f"l{i}", layer["mixer"], layer["mlp"]["router"]
        h = _rms(x, eps) * (1 + w(p + ".norm1"))
        if layer["type"] == "attention":
            q, k, v = ((h @ w(f"{p}.mix.{n}").T).view(T, -1, m["dim"]) for n in "qkv")
            q, k = (_turn_pairs(_rms(t, eps) * w(f"{p}.mix.{n}.norm"), *_yarn_frequencies(m["rot"]))
                    for n, t in (("q", q), ("k", k)))
            o = _attend(q, k, v, m["scale"], m["mask"]["size"], w(p + ".mix.sink"))
            y = o.reshape(T, -1) @ w(p + ".mix.o").T
        else:
            y = _mlstm(h, w, p + ".mix", m, eps)
        h = _rms(x, eps) * (1 + w(p + ".norm2"))
        s = torch.softmax(h @ w(p + ".mlp.router").T, -1)
        chosen = torch.topk(s + w(p + ".mlp.correction"), r["top"], -1).indices
        g = s.gather(-1, chosen)
        g = torch.zeros_like(s).scatter(-1, chosen, g / (g.sum(-1, keepdim=True) + 1e-20))
        y = y + _gated(h, w, p + ".mlp.shared") + g[:, r["experts"]:].sum(-1, keepdim=True) * h
        for e in range(r["experts"]):
            at = g[:, e].nonzero()[:, 0]
            if len(at):
                y[at] += g[at, e, None] * _gated(h[at], w, f"{p}.mlp.e{e}")
        x = x + y
    return _rms(x, eps) * (1 + w("final.norm"))


def _turn_halves(x, rot):
    freq, mag = _yarn_frequencies(rot)
    cos, sin = (t * mag for t in _angles(freq, x.shape[0]))
    u, v = x.split(len(freq), -1)
    return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)


def _latent(h, w, p, m, eps):
    T, H, d, rank = h.shape[0], m["heads"], m["dim"], m["kv_rank"]
    q = ((_rms(h @ w(p + "dq").T, eps) * w(p + "dq.norm")) @ w(p + "uq").T).view(T, H, -1)
    q = torch.cat([q[..., :d], _turn_halves(q[..., d:], m["rot"])], -1)
    rows = h @ w(p + "dkv").T
    c, kr = _rms(rows[:, :rank], eps) * w(p + "dkv.norm"), _turn_halves(rows[:, None, rank:], m["rot"])
    k = torch.cat([(c @ w(p + "uk").T).view(T, H, d), kr.expand(T, H, -1)], -1)
    o = _attend(q, k, (c @ w(p + "uv").T).view(T, H, -1), m["scale"]).reshape(T, -1)
    return (o * torch.sigmoid(h @ w(p + "g").T)) @ w(p + "o").T


def _short_conv(x, taps):
    n = taps.shape[1]
    padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    return sum(taps[:, j] * padded[j:j + len(x)] for j in range(n))


def _bucket(n, buckets, far):
    half = buckets // 2
    if n < half:
        return n
    return min(buckets - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (buckets - half)))


def _near(h, w, p, m, eps):
    T, d = h.shape[0], m["dim"]
    q, k, v = (_short_conv(h @ w(p + n).T, w(p + n + ".conv")).view(T, -1, d) for n in "qkv")
    bias = w(p + "rel")[[_bucket(n, m["buckets"], m["bias_max"]) for n in range(T)]]
    o = _attend(_rms(q, eps), _rms(k, eps), v, m["scale"], m["mask"]["size"], keep=m["mask"]["keep_first"], bias=bias)
    return (o * torch.sigmoid(h @ w(p + "g").T)[..., None]).reshape(T, -1) @ w(p + "o").T


def _memory(h, w, p, m, eps):
    T, H, G, dk, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (F.silu(_short_conv(h @ w(p + n).T, w(p + n + ".conv"))) for n in "qkv")
    q, k = (t.view(T, G, dk) * torch.rsqrt(t.view(T, G, dk).pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = (t.repeat_interleave(H // G, 1) for t in (q * dk ** -0.5, k))
    v, beta = v.view(T, H, dv), torch.sigmoid(h @ w(p + "b").T)
    z = (h @ w(p + "a1").T) @ w(p + "a2").T + w(p + "dt_bias")
    g = torch.exp(-torch.exp(w(p + "A_log"))[:, None] * F.softplus(z, threshold=1e9).view(T, H, dk))
    S, out = h.new_zeros(H, dk, dv), h.new_empty(T, H, dv)
    for t in range(T):
        S = g[t][:, :, None] * S
        u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None, :], S)[:, 0])
        S = torch.baddbmm(S, k[t][:, :, None], u[:, None, :])
        out[t] = torch.bmm(q[t][:, None, :], S)[:, 0]
    o = (_rms(out, eps) * w(p + "norm")).reshape(T, H * dv)
    return (o * torch.sigmoid((h @ w(p + "g1").T) @ w(p + "g2").T)) @ w(p + "o").T


def _limited(g, u, limit):
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def _depolix_rows(cfg, w, ids):
    eps = cfg["norm"]["eps"]
    x = w("embed")[ids] * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = f"l{i}.mix.", layer["mixer"], layer["mlp"]
        h = _rms(x, eps) * (1 + w(f"l{i}.norm1"))
        if layer["type"] == "latent_attention":
            y = _latent(h, w, p, m, eps)
        else:
            y = 0.5 * (_rms(_near(h, w, p + "left.", m["left"], eps), eps) * w(p + "left.out")
                       + _rms(_memory(h, w, p + "right.", m["right"], eps), eps) * w(p + "right.out"))
        p = f"l{i}.mlp."
        if mlp["kind"] == "dense":
            a = _limited(h @ w(p + "gate").T + w(p + "gate.b"), h @ w(p + "up").T + w(p + "up.b"), mlp["limit"])
            y = y + a @ w(p + "down").T + w(p + "down.b")
        else:
            best = torch.topk(h @ w(p + "router").T + w(p + "router.b"), mlp["router"]["top"], -1)
            share = torch.softmax(best.values, -1)
            for e in range(mlp["router"]["experts"]):
                at, j = (best.indices == e).nonzero(as_tuple=True)
                if len(at):
                    a = _limited(h[at] @ w(f"{p}e{e}.gate").T, h[at] @ w(f"{p}e{e}.up").T, mlp["expert"]["limit"])
                    y[at] += share[at, j, None] * (a @ w(f"{p}e{e}.down").T)
        x = x + cfg["residual_mult"] * y
    return _rms(x, eps) * (1 + w("final.norm"))


@torch.no_grad()
def exact(case, seed):
    cfg = _config(case)
    runs, singles = _sizes(case)
    seqs = _sequences(case, seed)
    weights = _drawn(case, seed)[1]
    wide: dict[str, torch.Tensor] = {}

    def w(name):
        if name not in wide:
            wide[name] = weights[name].double()
        return wide[name]

    scale, cap, head = 1.0, None, "head"
    if case["model"].startswith("rudorax"):
        rows_of, cap = _rudorax_rows, cfg["logit_softcap"]
    elif case["model"].startswith("depolix"):
        rows_of, scale = _depolix_rows, cfg["logit_scale"]
    else:
        rows_of = _llama_rows
        head = "model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"

    def logits(rows):
        z = scale * (rows @ w(head).T)
        return cap * torch.tanh(z / cap) if cap else z

    first, asked, picked = [], [], []
    for i, s in enumerate(seqs):
        end = sum(runs[i]) if i < len(runs) else singles[i - len(runs)]
        if not case["runs"]:                       # whole runs, or a single token behind its context
            first.append(logits(rows_of(cfg, w, s[:end if i < len(runs) else end + 1])[-1:])[0])
            continue
        # the tokens of a longer run are fed back, and a tie that falls otherwise changes all behind it
        given = s if case["steps"] == 1 else s[:end + 2]
        z = logits(rows_of(cfg, w, given)[max(end - 1, 0):])
        first.append(z[0])
        asked.append(z[1])
        picked.append(z[2:].argmax(-1))
    if not case["runs"]:
        return {"logits": torch.stack(first)}
    out = {"logits": torch.stack(asked), "tokens": None}
    if case["steps"] == 1 and not case["sampled"]:
        out["tokens"] = torch.stack(picked, 1)
    return dict(out, prompt_logits=torch.stack(first)) if runs else out
