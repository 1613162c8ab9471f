"""The work that programs have this package do, as cases that can be timed: a token at a time, verification of drafted tokens, batches
that decode, prompts from a chat line to the longest batch the engine admits, and whole requests and traces of the decoders that bring
their own config.json.  Every case goes through ModelRunner.run (what the engine's steps call) or TraceEngine.step (what bin/trace_run
calls), on published layer shapes with a reduced number of layers and random weights.

A case's keys: path, model, layers, batch, tokens (the longest prompt or context; the others are shorter, see _lengths), prefix (prompt
tokens whose pages are already cached), k (drafted tokens), steps (decoded tokens), portion (prompt tokens a trace feeds per step)."""
from __future__ import annotations

import math
import random
from dataclasses import replace

import torch

from ssd_amd.config import Config
from ssd_amd.engine.model_runner import ModelRunner
from ssd_amd.engine.sequence import Sequence
from ssd_amd.engine.trace_engine import TraceEngine
from ssd_amd.model_config import PRESETS, FatulixConfig, TumudraConfig

PAGE = 256                      # the engine's default page
F64 = torch.float64
DEV = "cuda"


def listed() -> list[dict]:
    return [
        # one chat, one token: the draft model's every step, and decoding without speculation
        dict(name="token", path="decode", model="llama-3.2-1b", layers=16, batch=1, tokens=300),
        # the target's step of synchronous speculation: one chat, k + 1 rows
        dict(name="verify", path="verify", model="llama-3.1-8b", layers=8, batch=1, tokens=700, k=6),
        # the same for four chats of a model with q / k norms: 32 rows
        dict(name="verify_batch", path="verify", model="qwen3-32b", layers=2, batch=4, tokens=1500, k=7),
        # a server's batch, contexts from a few dozen to a few thousand tokens
        dict(name="decode_batch", path="decode", model="llama-3.1-8b", layers=4, batch=48, tokens=3000),
        # the first token of a short prompt on the largest model
        dict(name="first_token", path="prefill", model="llama-3.1-70b", layers=2, batch=1, tokens=128, prefix=0),
        # a batch of ragged prompts on a small model
        dict(name="prompts_small", path="prefill", model="llama-3.2-1b", layers=16, batch=7, tokens=900, prefix=0),
        # ragged prompts behind a shared, cached system prompt
        dict(name="prompts_prefix", path="prefill", model="llama-3.1-8b", layers=4, batch=3, tokens=1501, prefix=512),
        # one document as long as the engine's default token budget
        dict(name="document", path="prefill", model="llama-3.1-8b", layers=2, batch=1, tokens=16384, prefix=0),
        # whole requests of a decoder with attention and recurrent layers: prompts, then tokens
        dict(name="requests", path="generate", model="tumudra-4096", layers=4, batch=4, tokens=1800, steps=12),
        # a trace in true fp32 through routed experts: prompt portions beside single tokens
        dict(name="trace_fp32", path="trace", model="fatulix-2048", layers=4, batch=3, tokens=1000, portion=512, steps=6),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    path = rng.choice(["decode", "decode", "verify", "prefill", "prefill", "prefill", "generate", "trace"])
    if path == "generate":
        return dict(path=path, model=rng.choice(["tumudra-2048", "tumudra-4096"]), layers=4, batch=_log(rng, 1, 4), tokens=_log(rng, 40, 1800),
                    steps=_log(rng, 2, 12))
    if path == "trace":
        return dict(path=path, model="fatulix-2048", layers=rng.randint(1, 4), batch=rng.randint(1, 3), tokens=_log(rng, 30, 1000),
                    portion=_log(rng, 30, 600), steps=_log(rng, 2, 6))
    model = rng.choice(["llama-3.2-1b", "llama-3.2-3b", "llama-3.1-8b", "qwen3-0.6b", "qwen3-8b"] if path != "verify" else
                       ["llama-3.1-8b", "llama-3.1-70b", "qwen3-8b", "qwen3-32b"])
    case = dict(path=path, model=model, layers=rng.randint(2, 4))
    if path == "decode":
        return dict(case, batch=_log(rng, 1, 64), tokens=_log(rng, 64, 4000))
    if path == "verify":
        return dict(case, batch=_log(rng, 1, 8), tokens=_log(rng, 64, 3000), k=rng.randint(1, 7))
    batch = _log(rng, 1, 8)
    return dict(case, batch=batch, tokens=_log(rng, 24, 8192 // batch), prefix=rng.choice([0, 0, 256, 768]))


def _lengths(n: int, top: int) -> list[int]:
    """n lengths up to `top` (the first), the others spread over a factor of sixteen: part of a case, the same for every seed."""
    r = random.Random(n * 1000003 + top)
    return [top] + [_log(r, max(1, top // 16), top) for _ in range(n - 1)]


# ------------------------------------------------------------------------------------------------------------------
# models and weights: matrices N(0, 1 / inputs), norm weights near one, as trained models' activations have unit scale
# ------------------------------------------------------------------------------------------------------------------
def _native(case: dict) -> dict:
    """config.json of the decoders that bring their own: published-size layers of width 2048 or 4096."""
    kind, width = case["model"].split("-")
    W, L = int(width), case["layers"]
    H, G = W // 128, W // 512
    if kind == "fatulix":
        layer = {"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": 64, "vdim": 128, "diff": 0.25, "scale": 64 ** -0.5},
                 "mlp": {"kind": "moe", "expert": {"ff": 3 * W // 4}, "router": {"experts": 8, "top": 2}, "shared": {"ff": 3 * W // 2}}}
        return {"vocab": 32000, "width": W, "norm": {"eps": 1e-5}, "layers": [layer] * L, "loop": {"start": 0, "stop": 0, "times": 1}}
    mlp = {"kind": "dense", "ff": {2048: 7424, 4096: 14720}[W]}
    att = {"heads": H, "kv_heads": G, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 5e5, "dims": 128}}
    left = {**att, "rot": {"base": 1e6, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}, "mask": {"size": 1024}}
    layers = [{"type": "parallel", "mixer": {"left": left, "right": {"heads": H // 2, "dim": 128, "vdim": 128, "gate_cap": 15.0}}, "mlp": mlp},
              {"type": "attention", "mixer": att, "mlp": mlp},
              {"type": "retention", "mixer": {"heads": H, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** -(3 + 5 * h / H) for h in range(H)],
                                              "rot": {"base": 1e6, "dims": 128}}, "mlp": mlp},
              {"type": "attention", "mixer": {**att, "kv_from": 1}, "mlp": mlp}]
    return {"vocab": 32000, "width": W, "norm": {"eps": 1e-5}, "embedding": {"scale": 4.0}, "layers": layers[:L]}


def _model_config(case: dict):
    if case["path"] == "generate":
        return TumudraConfig.from_json(_native(case))
    if case["path"] == "trace":
        return FatulixConfig.from_json(_native(case))
    return replace(PRESETS[case["model"]], num_layers=case["layers"])


def _shapes(case: dict) -> list[tuple[str, tuple]]:
    """(name, shape) of every tensor of the model's checkpoint."""
    if case["path"] == "trace":
        c = _native(case)
        W, out = c["width"], [("embed", (c["vocab"], c["width"]))]
        for i, lc in enumerate(c["layers"]):
            p, m, ml = f"l{i}.", lc["mixer"], lc["mlp"]
            D, ff, sff = m["dim"], ml["expert"]["ff"], ml["shared"]["ff"]
            out += [(p + n, (W,)) for n in ("norm1", "norm1b", "norm2", "norm2b")]
            out += [(p + "mix.q", (m["heads"] * 2 * D, W)), (p + "mix.k", (m["kv_heads"] * 2 * D, W)), (p + "mix.v", (m["kv_heads"] * m["vdim"], W)),
                    (p + "mix.g", (m["heads"], W)), (p + "mix.o", (W, m["heads"] * m["vdim"])), (p + "mix.q.norm", (D,)), (p + "mix.k.norm", (D,))]
            out += [(p + "mix." + n, (D,)) for n in ("lq1", "lk1", "lq2", "lk2")]
            out += [(p + f"mlp.e{e}.{n}", s) for e in range(ml["router"]["experts"]) for n, s in (("up", (ff, W)), ("down", (W, ff)))]
            out += [(p + "mlp.router", (ml["router"]["experts"], W)), (p + "mlp.shared.up", (sff, W)), (p + "mlp.shared.down", (W, sff))]
        return out + [("final.norm", (W,)), ("head", (c["vocab"], W))]
    if case["path"] == "generate":
        c = _native(case)
        W, out = c["width"], [("embed", (c["vocab"], c["width"]))]
        for i, lc in enumerate(c["layers"]):
            p, m, bias = f"l{i}.mix.", lc["mixer"], lc["type"] == "attention"
            out.append((f"l{i}.norm1", (W,)))
            if lc["type"] != "retention":
                a, q = (m, p) if bias else (m["left"], p + "left.")
                mats = [("q", a["heads"] * a["dim"], W), ("o", W, a["heads"] * a["vdim"])]
                out.append((q + "q.norm", (a["dim"],)))
                if a.get("kv_from") is None:
                    mats += [("k", a["kv_heads"] * a["dim"], W), ("v", a["kv_heads"] * a["vdim"], W)]
                    out.append((q + "k.norm", (a["dim"],)))
                out += [(q + n, (r, k)) for n, r, k in mats] + ([(q + n + ".b", (r,)) for n, r, _ in mats] if bias else [])
            if not bias:
                a, q = (m, p) if lc["type"] == "retention" else (m["right"], p + "right.")
                nk, nv = a["heads"] * a["dim"], a["heads"] * a["vdim"]
                out += [(q + "q", (nk, W)), (q + "k", (nk, W)), (q + "v", (nv, W)), (q + "g", (nv, W)), (q + "o", (W, nv))]
                if lc["type"] == "parallel":
                    out += [(q + "norm", (nv,)), (p + "left.out", (W,)), (p + "right.out", (W,))]
                    out += [t for n in "if" for t in ((q + n, (a["heads"], W)), (q + n + ".b", (a["heads"],)))]
            ff = lc["mlp"]["ff"]
            out += [(f"l{i}.norm2", (W,)), (f"l{i}.mlp.up", (ff, W)), (f"l{i}.mlp.down", (W, ff))]
        return out + [("final.norm", (W,)), ("head", (c["vocab"], W))]
    c = _model_config(case)
    h, hd, I, V = c.hidden_size, c.head_dim, c.intermediate_size, c.vocab_size
    out = [("model.embed_tokens.weight", (V, h))]
    for i in range(c.num_layers):
        p = f"model.layers.{i}."
        out += [(p + "input_layernorm.weight", (h,)), (p + "self_attn.qkv_proj.weight", ((c.num_heads + 2 * c.num_kv_heads) * hd, h))]
        if c.qk_norm:
            out += [(p + "self_attn.q_norm.weight", (hd,)), (p + "self_attn.k_norm.weight", (hd,))]
        out += [(p + "self_attn.o_proj.weight", (h, c.num_heads * hd)), (p + "post_attention_layernorm.weight", (h,)),
                (p + "mlp.gate_up_proj.weight", (2 * I, h)), (p + "mlp.down_proj.weight", (h, I))]
    out.append(("model.norm.weight", (h,)))
    return out + ([] if c.tie_word_embeddings else [("lm_head.weight", (V, h))])


def _weights(case: dict, seed: int):
    """(name, bf16 tensor) pairs, one after the other."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    for name, shape in _shapes(case):
        t = torch.randn(*shape, generator=g, device=DEV)
        if name.endswith((".lq1", ".lk1", ".lq2", ".lk2")):
            t = 0.2 * t
        elif name.endswith("f.b"):                      # forget gates from a few tokens to hundreds
            t = 2.0 + t
        elif name.endswith(".b"):
            t = 0.2 * t
        elif len(shape) == 1:
            t = 1.0 + 0.1 * t
        elif "embed" not in name or name.startswith("model."):
            # (a tied embedding is the head as well; the first norm makes its scale of no account)
            t = t / math.sqrt(shape[-1])
        yield name, t.to(torch.bfloat16)


def _tokens(case: dict, seed: int, n: int) -> list[int]:
    g = torch.Generator().manual_seed(7919 * seed + n)
    return torch.randint(0, _model_config(case).vocab_size, (n,), generator=g).tolist()


# ------------------------------------------------------------------------------------------------------------------
# the requests of a case: token lists, and where their pages lie (the shared prefix first, then one run of pages each)
# ------------------------------------------------------------------------------------------------------------------
def _requests(case: dict, seed: int) -> list[list[int]]:
    """Every request's tokens, those of the pass itself included."""
    extra = {"decode": 1, "verify": case.get("k", 0) + 1, "generate": case.get("steps", 0), "trace": case.get("steps", 0)}.get(case["path"], 0)
    prefix = _tokens(case, seed, case.get("prefix", 0))
    out, at = [], 1
    for n in _lengths(case["batch"], case["tokens"]):
        out.append(prefix + _tokens(case, seed + 31 * at, n + extra))
        at += 1
    return out


def _tables(case: dict, requests) -> tuple[list[list[int]], int]:
    shared = case.get("prefix", 0) // PAGE
    tables, nxt = [], shared
    for r in requests:
        own = -(-len(r) // PAGE) - shared
        tables.append(list(range(shared)) + list(range(nxt, nxt + own)))
        nxt += own
    return tables, nxt


def _request(tokens, table, cached: int, slot: int = -1) -> Sequence:
    s = Sequence(tokens)
    s.block_table, s.num_cached_tokens, s.state_slot = list(table), cached, slot
    return s


def prepare(case: dict, seed: int) -> dict:
    cfg, path = _model_config(case), case["path"]
    requests = _requests(case, seed)
    if path == "trace":
        def runner(config):
            return ModelRunner(config, cfg, is_draft=False, device=torch.device("cuda", 0), weight_source=_weights(case, seed),
                               num_kvcache_blocks=config.num_kvcache_blocks)
        room = sum(-(-len(r) // 64) * 64 for r in requests)
        engine = TraceEngine("synthetic", dtype="float32", max_tokens=room, max_live=case["batch"], block_size=64, runner_factory=runner,
                             hf_config=cfg)
        return dict(case=case, engine=engine, plan=_plan(case, requests))
    tables, pages = _tables(case, requests)
    longest = -(-max(len(r) for r in requests) // PAGE) * PAGE
    new = max(longest, sum(len(r) for r in requests) if path in ("prefill", "generate") else 0)
    spec = dict(speculate=True, draft="draft", draft_hf_config=cfg, speculate_k=case["k"]) if path == "verify" else {}
    config = Config("synthetic", hf_config=cfg, kvcache_block_size=PAGE, max_num_seqs=case["batch"], max_model_len=longest,
                    max_num_batched_tokens=new, num_kvcache_blocks=pages, **spec)
    Sequence.block_size = PAGE
    runner = ModelRunner(config, cfg, is_draft=False, device=torch.device("cuda", 0), weight_source=_weights(case, seed), num_kvcache_blocks=pages)
    state = dict(case=case, runner=runner)
    if path == "generate":
        return dict(state, prompts=[r[:len(r) - case["steps"]] for r in requests], given=[r[len(r) - case["steps"]:] for r in requests],
                    tables=tables)
    if path == "prefill":
        prefix = case["prefix"]
        if prefix:
            runner.run([_request(requests[0][:prefix], tables[0], 0)], True)
        return dict(state, seqs=[_request(r, t, prefix) for r, t in zip(requests, tables)])
    old = [len(r) - (case.get("k", 0) + 1) for r in requests]           # tokens whose keys and values are there already
    for r, t, n in zip(requests, tables, old):
        runner.run([_request(r[:n], t, 0)], True)
    return dict(state, seqs=[_request(r, t, n) for r, t, n in zip(requests, tables, old)])


def _plan(case: dict, requests) -> list:
    """Steps of a trace: request r comes in at step r; a step brings the next portion of its prompt or one more token; its last row's
    logits are asked for."""
    at, steps, done = [0] * len(requests), [], 0
    while done < len(requests):
        entries, end = [], []
        for i, r in enumerate(requests):
            if i > len(steps) or at[i] >= len(r):
                continue
            prompt = len(r) - case["steps"]
            n = min(case["portion"], prompt - at[i]) if at[i] < prompt else 1
            entries.append({"id": str(i), "tokens": r[at[i]:at[i] + n], "want": [n - 1]})
            at[i] += n
            if at[i] >= len(r):
                end.append(str(i))
                done += 1
        steps.append((entries, end))
    return steps


def run(state: dict):
    path = state["case"]["path"]
    if path == "trace":
        return [state["engine"].step(entries, end) for entries, end in state["plan"]]
    runner = state["runner"]
    if path == "decode":
        return runner.run(state["seqs"], False, True, True)[1]
    if path == "verify":
        return runner.run(state["seqs"], False, False)
    if path == "prefill":
        return dict(logits=runner.run(state["seqs"], True, True, True)[1], kv=runner.model.kv_cache)
    seqs = [_request(p, t, 0, i) for i, (p, t) in enumerate(zip(state["prompts"], state["tables"]))]
    out = [runner.run(seqs, True, True, True)[1].clone()]
    for j in range(state["case"]["steps"]):
        for s, g in zip(seqs, state["given"]):
            s.append_token(g[j])
            s.num_cached_tokens = len(s) - 1
        out.append(runner.run(seqs, False, True, True)[1].clone())
    return torch.stack(out)


# ------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------------------------
def work(case: dict) -> dict:
    """Bytes: every matrix that has rows to work on once (once per step where steps follow each other), the keys and values of the
    context once, those of new tokens and the logits written.  Operations: the products, two per weight and row, and attention's two
    per key and channel pair."""
    path, W = case["path"], 4 if case["path"] == "trace" else 2
    size = {n: math.prod(s) for n, s in _shapes(case)}
    body = sum(v for n, v in size.items() if "embed" not in n and "head" not in n)
    lens = _lengths(case["batch"], case["tokens"])
    B = len(lens)
    if path in ("decode", "verify", "prefill"):
        c = _model_config(case)
        head, kv = c.vocab_size * c.hidden_size, 2 * c.num_kv_heads * c.head_dim * c.num_layers
        att = 4 * c.num_heads * c.head_dim * c.num_layers
        q = {"decode": 1, "verify": case.get("k", 0) + 1}.get(path)
        pre = case.get("prefix", 0)
        rows, out = (q * B, q * B) if q else (sum(lens), B)
        old = sum(lens) if q else pre
        pairs = sum(q * n + q * (q + 1) // 2 for n in lens) if q else sum(n * pre + n * (n + 1) // 2 for n in lens)
        return dict(bytes=W * (body + head + kv * (old + rows) + out * c.vocab_size), flops=2 * (rows * body + out * head) + att * pairs)
    c = _native(case)
    head = size["head"]
    if path == "generate":
        n, H = case["steps"], c["width"] // 128
        rows = sum(lens) + B * n
        kv = 2 * (c["width"] // 4)                          # key and value entries of a token in one attention layer
        window = lambda k: min(k, 1024)
        kinds = [l["type"] for l in c["layers"]]
        reads = sum(kinds.count("attention") * k + kinds.count("parallel") * window(k) for x in lens for k in range(x, x + n))
        pairs = sum(kinds.count("attention") * k + kinds.count("parallel") * window(k) for x in lens for k in range(1, x + n + 1))
        scans = 6 * 128 * 128 * (kinds.count("retention") * H + kinds.count("parallel") * H // 2)
        return dict(bytes=2 * ((n + 1) * (body + head) + kv * (reads + 2 * rows) + (n + 1) * B * c["vocab"]),
                    flops=2 * (rows * body + (n + 1) * B * head) + 4 * c["width"] * pairs + scans * rows)
    experts = sum(v for n, v in size.items() if ".e" in n)
    steps = _plan(case, [[0] * (x + case["steps"]) for x in lens])
    E, top = 8, 2
    nbytes = flops = 0
    seen = [0] * B
    for entries, _ in steps:
        rows = sum(len(e["tokens"]) for e in entries)
        nbytes += body - experts + head + experts * min(E, rows * top) // E + len(entries) * c["vocab"]
        flops += 2 * (rows * (body - experts + experts * top // E) + len(entries) * head)
        for e in entries:
            i, n = int(e["id"]), len(e["tokens"])
            nbytes += 2 * (c["width"] // 4) * case["layers"] * (seen[i] + n)
            flops += 6 * c["width"] * case["layers"] * (seen[i] * n + n * (n + 1) // 2)
            seen[i] += n
    return dict(bytes=W * nbytes, flops=flops)


def tolerance(case: dict):
    """fp32 sums in another order, or bf16 rows that such sums round to their neighbour, carried through the layers.  Against 64 bits
    the outputs are 2e-6 .. 3e-6 off in fp32, 3e-3 with an fp32 residual row and 6e-3 .. 1.5e-2 with a bf16 one; two orders of
    summation differ by less than two such errors."""
    if case["path"] == "trace":
        return dict(rel=1e-5, max=1e-4)
    return dict(rel=0.01, max=0.1) if case["path"] == "generate" else dict(rel=0.025, max=0.25)


# ------------------------------------------------------------------------------------------------------------------
# the same in 64 bits, one function per kind of model: whole sequences, no cache
# ------------------------------------------------------------------------------------------------------------------
def _norm(x, w=None, eps=1e-5):
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w.double()


def _lin(x, w, bias=None):
    y = x @ w.double().T
    return y if bias is None else y + bias.double()


def _turn(x, base, dims, interleaved=False, scaling=None):
    """Rotary positions 0 .. T - 1 of x [T, heads, D]."""
    f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=x.device) / dims)
    if scaling:
        turns = scaling["original"] * f / (2.0 * math.pi)
        keep = ((turns - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0.0, 1.0)
        f = (1.0 - keep) * f / scaling["factor"] + keep * f
    t = torch.arange(x.shape[0], dtype=F64, device=x.device).view(-1, 1, 1) * f
    c, s = torch.cos(t), torch.sin(t)
    a, b = (x[..., 0:dims:2], x[..., 1:dims:2]) if interleaved else (x[..., :dims // 2], x[..., dims // 2:dims])
    a, b = a * c - b * s, b * c + a * s
    y = torch.stack([a, b], -1).flatten(-2) if interleaved else torch.cat([a, b], -1)
    return torch.cat([y, x[..., dims:]], -1)


def _attend(q, k, v, scale, window=0):
    """q [T, H, D], k [T, G, D], v [T, G, Dv] -> [T, H, Dv]; some query rows at a time."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=F64, device=q.device)
    step = max(1, min(T, (1 << 28) // (T * H // G)))
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        for a in range(0, T, step):
            b = min(T, a + step)
            s = torch.matmul(q[a:b, hs].reshape(-1, q.shape[2]), k[:b, g].T.contiguous()).view(b - a, H // G, b) * scale
            d = torch.arange(a, b, device=q.device).view(-1, 1) - torch.arange(b, device=q.device).view(1, -1)
            hide = (d < 0) | (d >= window) if window else d < 0
            p = torch.softmax(s.masked_fill(hide.unsqueeze(1), -math.inf), -1)
            out[a:b, hs] = torch.matmul(p.view(-1, b), v[:b, g].contiguous()).view(b - a, H // G, -1)
    return out


def _llama(case, w, tokens, keep):
    """Logits of the rows from `keep` on, and every layer's keys and values [T, G, hd]."""
    c = _model_config(case)
    T, H, G, hd, eps = len(tokens), c.num_heads, c.num_kv_heads, c.head_dim, c.rms_norm_eps
    x, kvs = w["model.embed_tokens.weight"][torch.tensor(tokens, device=DEV)].double(), []
    for i in range(c.num_layers):
        p = f"model.layers.{i}."
        y = _lin(_norm(x, w[p + "input_layernorm.weight"], eps), w[p + "self_attn.qkv_proj.weight"]).view(T, H + 2 * G, hd)
        q, k, v = y[:, :H], y[:, H:H + G], y[:, H + G:]
        if c.qk_norm:
            q, k = _norm(q, w[p + "self_attn.q_norm.weight"], eps), _norm(k, w[p + "self_attn.k_norm.weight"], eps)
        q, k = _turn(q, c.rope_theta, hd), _turn(k, c.rope_theta, hd)
        kvs.append((k, v))
        if i == c.num_layers - 1 and keep > 0:          # nothing reads the earlier rows after the last layer's keys and values
            o = _attend_rows(q, k, v, hd ** -0.5, keep)
            x = x[keep:]
        else:
            o = _attend(q, k, v, hd ** -0.5)
        x = x + _lin(o.flatten(1), w[p + "self_attn.o_proj.weight"])
        gate, up = _lin(_norm(x, w[p + "post_attention_layernorm.weight"], eps), w[p + "mlp.gate_up_proj.weight"]).chunk(2, -1)
        x = x + _lin(gate * torch.sigmoid(gate) * up, w[p + "mlp.down_proj.weight"])
        del gate, up
    return _lin(_norm(x, w["model.norm.weight"], eps), w.get("lm_head.weight", w["model.embed_tokens.weight"])), kvs


def _attend_rows(q, k, v, scale, first):
    """_attend of the rows from `first` on."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    q = q[first:]
    s = torch.einsum("thd,khd->htk", q, k.repeat_interleave(H // G, 1)) * scale
    d = torch.arange(first, T, device=q.device).view(-1, 1) - torch.arange(T, device=q.device).view(1, -1)
    return torch.einsum("htk,khd->thd", torch.softmax(s.masked_fill(d < 0, -math.inf), -1), v.repeat_interleave(H // G, 1))


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.double()


def _decayed(q, k, v, log_weight):
    """sum over j <= t of e^log_weight[t, j, h] <q_t, k_j> v_j, a head at a time: a linear recurrence written out."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=F64, device=q.device)
    for h in range(q.shape[1]):
        out[:, h] = (torch.matmul(q[:, h], k[:, h].T.contiguous()) * torch.exp(log_weight(h)).tril()) @ v[:, h]
    return out


def _tumudra(case, w, tokens):
    c = _native(case)
    T, W, eps = len(tokens), c["width"], c["norm"]["eps"]
    x, kvs = w["embed"][torch.tensor(tokens, device=DEV)].double() * c["embedding"]["scale"], {}
    back = lambda f: f.view(-1, 1) - f.view(1, -1)

    def attention(i, p, m, inter):
        bias = lambda n: w.get(p + n + ".b")
        turn = lambda t: _turn(t, m["rot"]["base"], m["rot"]["dims"], inter, m["rot"].get("scaling"))
        q = turn(_norm(_lin(x, w[p + "q"], bias("q")).view(T, m["heads"], m["dim"]), w[p + "q.norm"], eps))
        if m.get("kv_from") is None:
            k = turn(_norm(_lin(x, w[p + "k"], bias("k")).view(T, m["kv_heads"], m["dim"]), w[p + "k.norm"], eps))
            kvs[i] = k, _lin(x, w[p + "v"], bias("v")).view(T, m["kv_heads"], m["vdim"])
        o = _attend(q, *kvs[m.get("kv_from", i)], m["scale"], (m.get("mask") or {}).get("size", 0))
        return _lin(o.flatten(1), w[p + "o"], bias("o"))

    def linear(p, m):
        H, D = m["heads"], m["dim"]
        q, k = (_lin(x, w[p + n]).view(T, H, D) for n in "qk")
        return q, k, _lin(x, w[p + "v"]).view(T, H, -1), _lin(x, w[p + "g"]), H, D

    def retention(p, m):
        q, k, v, g, H, D = linear(p, m)
        turn = lambda t: _turn(t, m["rot"]["base"], m["rot"]["dims"])
        pos = torch.arange(T, dtype=F64, device=DEV)
        o = _decayed(turn(q), turn(k) * D ** -0.5, v, lambda h: back(pos) * math.log(m["decay"][h]))
        return _lin(_norm(o, None, eps).flatten(1) * g * torch.sigmoid(g), w[p + "o"])

    def memory(p, m):
        q, k, v, g, H, D = linear(p, m)
        q, cap = q * D ** -0.5, m["gate_cap"]
        gate = lambda n: cap * torch.tanh(_lin(x, w[p + n], w[p + n + ".b"]) / cap)
        i, f = gate("i"), torch.nn.functional.logsigmoid(gate("f")).cumsum(0)
        top = f + torch.cummax(i - f, 0).values.clamp(min=0.0)              # the running maximum, from 0
        o = _decayed(q, k, torch.cat([v, torch.ones_like(v[..., :1])], -1),
                     lambda h: (f[:, h] - top[:, h]).view(-1, 1) + (i[:, h] - f[:, h]).view(1, -1))
        o = o[..., :-1] / (torch.maximum(o[..., -1:].abs(), torch.exp(-top).unsqueeze(-1)) + 1e-6)
        return _lin(_norm(o, None, eps).flatten(1) * w[p + "norm"].double() * torch.sigmoid(g), w[p + "o"])

    for i, lc in enumerate(c["layers"]):
        p, m = f"l{i}.mix.", lc["mixer"]
        if lc["type"] == "parallel":
            y = 0.5 * (_norm(attention(i, p + "left.", m["left"], True), w[p + "left.out"], eps)
                       + _norm(memory(p + "right.", m["right"]), w[p + "right.out"], eps))
        else:
            y = attention(i, p, m, False) if lc["type"] == "attention" else retention(p, m)
        x = x + _layer_norm(y, w[f"l{i}.norm1"], eps)
        y = _lin(torch.relu(_lin(x, w[f"l{i}.mlp.up"])) ** 2, w[f"l{i}.mlp.down"])
        x = x + _layer_norm(y, w[f"l{i}.norm2"], eps)
    return _lin(_layer_norm(x, w["final.norm"], eps), w["head"])


def _fatulix(case, w, tokens):
    c = _native(case)
    T, eps = len(tokens), c["norm"]["eps"]
    x = w["embed"][torch.tensor(tokens, device=DEV)].double()
    expert = lambda t, p: _lin(torch.relu(_lin(t, w[p + "up"])) ** 2, w[p + "down"])
    for i, lc in enumerate(c["layers"]):
        p, m, ml = f"l{i}.mix.", lc["mixer"], lc["mlp"]
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        y = _norm(x, w[f"l{i}.norm1"], eps)
        q = _norm(_lin(y, w[p + "q"]).view(T, H, 2, D), w[p + "q.norm"], eps)
        k = _norm(_lin(y, w[p + "k"]).view(T, G, 2, D), w[p + "k.norm"], eps)
        v = _lin(y, w[p + "v"]).view(T, G, m["vdim"])
        a, b = (_attend(q[:, :, s], k[:, :, s], v, m["scale"]) for s in (0, 1))
        dot = lambda s: float(torch.exp((w[p + "lq" + s].double() * w[p + "lk" + s].double()).sum()))
        o = _norm(a - (dot("1") - dot("2") + m["diff"]) * b, None, eps) * (1.0 - m["diff"]) * torch.sigmoid(_lin(y, w[p + "g"])).unsqueeze(-1)
        x = x + _norm(_lin(o.flatten(1), w[p + "o"]), w[f"l{i}.norm1b"], eps)
        y, p = _norm(x, w[f"l{i}.norm2"], eps), f"l{i}.mlp."
        best, which = _lin(y, w[p + "router"]).topk(ml["router"]["top"], -1)
        share = torch.softmax(best, -1)
        z = expert(y, p + "shared.")
        for e in range(ml["router"]["experts"]):
            row, place = (which == e).nonzero(as_tuple=True)
            z[row] += share[row, place].unsqueeze(-1) * expert(y[row], p + f"e{e}.")
        x = x + _norm(z, w[f"l{i}.norm2b"], eps)
    return _lin(_norm(x, w["final.norm"], eps), w["head"])


@torch.inference_mode()
def exact(case: dict, seed: int):
    w, requests, path = dict(_weights(case, seed)), _requests(case, seed), case["path"]
    if path == "trace":
        logits = [_fatulix(case, w, r) for r in requests]
        at, out = [0] * len(requests), []
        for entries, _ in _plan(case, requests):
            rows = []
            for e in entries:
                i = int(e["id"])
                at[i] += len(e["tokens"])
                rows.append(logits[i][at[i] - 1])
            out.append(torch.stack(rows))
        return out
    if path == "generate":
        return torch.stack([_tumudra(case, w, r)[len(r) - case["steps"] - 1:] for r in requests], 1)
    if path != "prefill":
        q = case.get("k", 0) + 1
        return torch.cat([_llama(case, w, r, len(r) - q)[0] for r in requests])
    c = _model_config(case)
    tables, pages = _tables(case, requests)
    kv = torch.zeros(c.num_layers, 2, pages, c.num_kv_heads, PAGE, c.head_dim, dtype=F64, device=DEV)
    rows = []
    for r, table in zip(requests, tables):
        logits, kvs = _llama(case, w, r, len(r) - 1)
        rows.append(logits)
        for i, both in enumerate(kvs):
            for s, t in enumerate(both):
                for j, page in enumerate(table):
                    part = t[j * PAGE:(j + 1) * PAGE]
                    kv[i, s, page, :, :part.shape[0]] = part.transpose(0, 1)
    return dict(logits=torch.cat(rows), kv=kv)
