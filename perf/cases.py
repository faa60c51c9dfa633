"""The work a serving program gives this framework, as cases that can be timed.

Six kinds of case, each through the public entry points a program calls:

  forward   `Attention.forward`: one decode attention over a batch of cached sequences that share
            prefixes (the kernels' main path; the five benchmark configurations are of this kind)
  generate  the life of a batch on one cache: `add_seq` of every prompt (prefix matching and K/V
            copy-in), `decode_step` for every new token (append + attention, last chunks rolling
            over at different steps), `clear`
  beam      a beam search on one cache: `add_seq`, then per step `append_completion` for every
            beam, `remove_seq` of the beams that lost, `forward` over the survivors, `clear`
  layer     `LlamaChunkAttention`: a batch of prompts through the prefill branch (projections,
            rotary embedding, causal attention, insertion), decode steps, `clear`
  model     `AttentionOnlyLM`: prompts prefilled one by one as the scheduler does it, then decode
            iterations over the running batch; the continuation is given, the logits are returned
  ops       the operators around the attention call, as a layer uses them on a batch of tokens:
            `ops.fused_add_rms_norm`, then `ops.rotary_embedding`

Everything is float16, the only type the framework takes.  Inputs are drawn on the GPU from the
seed alone.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "chunk-attention_amd"))

from chunk_attn import Attention, ops  # noqa: E402
from chunk_attn import capi  # noqa: E402
from chunk_attn.llama_layer import LlamaChunkAttention  # noqa: E402
from chunk_attn.models.sequence import Sequence  # noqa: E402
from chunk_attn.models.tiny_lm import AttentionOnlyLM  # noqa: E402

D = 128                 # the head dimension the attention kernels take
DEV = "cuda:0"
HALF = torch.float16


# ---- the cases ---------------------------------------------------------------------------------

def _forward(name, batch, chunk, heads, root, group, per_group, unique, spread):
    """`batch` sequences = `root` tokens shared by all + `group` tokens shared by each `per_group`
    neighbours + private tokens, unique * (1 - spread) .. unique of them."""
    c = {"kind": "forward", "batch": batch, "chunk": chunk, "heads": heads, "root": root, "group": group,
         "per_group": per_group, "unique": unique, "spread": spread}
    return dict(c, name=name) if name else c


def _generate(name, batch, chunk, heads, root, unique, spread, steps):
    c = {"kind": "generate", "batch": batch, "chunk": chunk, "heads": heads, "root": root, "unique": unique,
         "spread": spread, "steps": steps}
    return dict(c, name=name) if name else c


def _beam(name, prompt, chunk, heads, width, steps):
    c = {"kind": "beam", "prompt": prompt, "chunk": chunk, "heads": heads, "width": width, "steps": steps}
    return dict(c, name=name) if name else c


def _layer(name, batch, prompt, heads, chunk, steps):
    c = {"kind": "layer", "batch": batch, "prompt": prompt, "heads": heads, "chunk": chunk, "steps": steps}
    return dict(c, name=name) if name else c


def _model(name, batch, root, unique, heads, layers, vocab, chunk, steps):
    c = {"kind": "model", "batch": batch, "root": root, "unique": unique, "heads": heads, "layers": layers,
         "vocab": vocab, "chunk": chunk, "steps": steps}
    return dict(c, name=name) if name else c


def _ops(name, tokens, hidden, neox):
    c = {"kind": "ops", "tokens": tokens, "hidden": hidden, "neox": neox}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a handful of chats on a small model (the class's default of 12 heads), a short common system
        # prompt: the smallest call, all latency
        _forward("chat-4", 4, 64, 12, 256, 0, 1, 100, 0.5),
        # the five benchmark configurations: 16 sequences with small chunks ...
        _forward("batch-16-c32", 16, 32, 32, 1024, 0, 1, 256, 0.0),
        # ... the headline workload ...
        _forward("batch-32", 32, 64, 32, 2048, 0, 1, 512, 0.0),
        # ... a prompt template and few-shot examples per task below it ...
        _forward("two-level-64", 64, 64, 32, 1024, 512, 8, 128, 0.0),
        # ... a large batch behind one long prompt ...
        _forward("batch-256", 256, 64, 32, 4096, 0, 1, 256, 0.0),
        # ... and the end of the sharing sweep at which nothing is shared: the largest call
        _forward("unshared-64", 64, 64, 32, 0, 0, 1, 4096, 0.0),
        # traffic as it comes: chunks of 128, prompts and answers of every length, 40 heads
        _forward("ragged-48-c128", 48, 128, 40, 1500, 0, 1, 900, 0.9),
        # a batch from admission to its last token
        _generate("generate-32", 32, 64, 32, 1024, 300, 0.4, 48),
        # beam search on one prompt
        _beam("beam-4", 1000, 64, 32, 4, 16),
        # a long prompt through one attention layer of a 7B model, then its first new token
        _layer("prefill-2048", 1, 2048, 32, 64, 1),
        # requests with a common system prompt through a small model
        _model("model-8", 8, 192, 60, 8, 4, 8000, 64, 16),
        # one layer's operators on a prefill batch
        _ops("ops-2048", 2048, 4096, True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    w = work(c)
    return max(w["bytes"], w["flops"] / 50)      # 50 operations a byte: what a large product costs beside a large copy


def draw(rng):
    kind = rng.choice(["forward"] * 6 + ["generate"] * 2 + ["beam", "layer", "model", "ops"])
    limit = max(_cost(c) for c in listed() if c["kind"] == kind or kind == "ops")
    while True:
        c = _draw(rng, kind)
        if _cost(c) <= limit:
            return c


def _draw(rng, kind):
    chunk = rng.choice([32, 64, 64, 128])
    if kind == "forward":
        batch = _log(rng, 1, 256)
        root = rng.choice([0, _log(rng, 64, 4096), _log(rng, 64, 4096), _log(rng, 64, 4096)])
        two = batch >= 8 and root > 0 and rng.random() < 0.3
        per_group = rng.randint(2, max(2, batch // 3)) if two else 1
        return _forward(None, batch, chunk, rng.choice([8, 12, 16, 32, 32, 32, 40]), root, _log(rng, 32, 1024) if two else 0,
                        per_group, _log(rng, 8, 4096), rng.choice([0.0, round(rng.uniform(0.1, 0.9), 2)]))
    if kind == "generate":
        return _generate(None, _log(rng, 2, 64), chunk, rng.choice([8, 12, 32]), _log(rng, 64, 2048), _log(rng, 16, 512),
                         round(rng.uniform(0.0, 0.9), 2), rng.randint(8, 60))
    if kind == "beam":
        return _beam(None, _log(rng, 64, 3000), chunk, rng.choice([8, 12, 32]), rng.randint(2, 8), rng.randint(8, 32))
    if kind == "layer":
        prompt = _log(rng, 64, 3000)
        return _layer(None, rng.randint(1, 8), prompt, rng.choice([8, 16, 32]), chunk, rng.randint(1, 8))
    if kind == "model":
        return _model(None, rng.randint(2, 12), _log(rng, 32, 512), _log(rng, 8, 256), rng.choice([2, 4, 8]), rng.randint(2, 4),
                      rng.choice([500, 4000, 8000]), chunk, rng.randint(4, 24))
    return _ops(None, _log(rng, 1, 16384), rng.choice([1024, 1536, 4096, 5120]), rng.random() < 0.7)


# ---- what a case consists of ---------------------------------------------------------------------

def _lengths(c):
    """Private tokens of every sequence: spread evenly over unique * (1 - spread) .. unique, in an
    order that has no pattern to it."""
    n = c["batch"]
    return [max(1, int(round(c["unique"] * (1.0 - c["spread"] * ((s * 0.6180339887) % 1.0))))) for s in range(n)]


def _attended(c, extra=0):
    """(tokens whose K/V one forward reads, tokens attended over all sequences), `extra` tokens
    after the prompts: whole chunks that several sequences share are read once."""
    chunk, read, pairs = c["chunk"], 0, 0
    lens, groups = _lengths(c), {}
    for s, n in enumerate(lens):
        groups.setdefault(s // c.get("per_group", 1) if c.get("group", 0) else s, []).append(n)
    batch, root, group = c["batch"], c["root"], c.get("group", 0)
    whole_root = root // chunk * chunk if batch > 1 else 0
    read += whole_root
    for members in groups.values():
        whole = (root + group) // chunk * chunk if group and len(members) > 1 else whole_root
        read += whole - whole_root
        for n in members:
            read += root + group + n + extra - whole
            pairs += root + group + n + extra
    return read, pairs


def _forward_work(c, extra=0):
    read, pairs = _attended(c, extra)
    h = c["heads"]
    return {"bytes": 4 * h * D * read + 4 * c["batch"] * h * D, "flops": 4 * h * D * pairs}


def _add(a, b):
    return {k: a[k] + b[k] for k in a}


def _layer_prefill_work(tokens, hidden, batch, heads):
    """Projections of batch x tokens rows and their causal attention."""
    rows = batch * tokens
    return {"bytes": 2 * 4 * hidden * hidden + 2 * 2 * rows * hidden + 2 * 2 * rows * hidden,
            "flops": 8 * rows * hidden * hidden + batch * 2 * heads * D * tokens * (tokens + 1)}


def _layer_decode_work(batch, hidden, heads, read, pairs):
    return {"bytes": 2 * 4 * hidden * hidden + 4 * batch * hidden + 4 * heads * D * read,
            "flops": 8 * batch * hidden * hidden + 4 * heads * D * pairs}


def work(case):
    c = case
    if c["kind"] == "forward":
        return _forward_work(c)
    if c["kind"] == "generate":
        read, _ = _attended(c)
        w = {"bytes": 8 * c["heads"] * D * read, "flops": 0}    # copy-in: K and V read and written
        for step in range(c["steps"]):
            w = _add(w, _forward_work(c, step + 1))
            w["bytes"] += 8 * c["batch"] * c["heads"] * D        # the new rows, read and written
        return w
    if c["kind"] == "beam":
        row = 4 * c["heads"] * D                                 # K and V of one token
        w = {"bytes": 2 * row * c["prompt"], "flops": 0}
        for step in range(c["steps"]):
            read = c["prompt"] // c["chunk"] * c["chunk"] + c["width"] * (c["prompt"] % c["chunk"] + step + 1)
            w["bytes"] += row * read + 3 * row * c["width"]
            w["flops"] += row * c["width"] * (c["prompt"] + step + 1)
        return w
    if c["kind"] == "layer":
        hidden = c["heads"] * D
        w = _layer_prefill_work(c["prompt"], hidden, c["batch"], c["heads"])
        for step in range(c["steps"]):
            n = c["batch"] * (c["prompt"] + step + 1)
            w = _add(w, _layer_decode_work(c["batch"], hidden, c["heads"], n, n))
        return w
    if c["kind"] == "model":
        hidden, head = c["heads"] * D, 2 * c["heads"] * D * c["vocab"]
        w = {"bytes": 0, "flops": 0}
        for _ in range(c["batch"]):
            for _ in range(c["layers"]):
                w = _add(w, _layer_prefill_work(c["root"] + c["unique"], hidden, 1, c["heads"]))
            w["bytes"] += head
            w["flops"] += head
        for step in range(c["steps"]):
            read, pairs = _attended(dict(c, spread=0.0), step + 1)
            for _ in range(c["layers"]):
                w = _add(w, _layer_decode_work(c["batch"], hidden, c["heads"], read, pairs))
            w["bytes"] += head
            w["flops"] += head * c["batch"]
        return w
    # activation and residual read and written, query and key read and written
    return {"bytes": 2 * 8 * c["tokens"] * c["hidden"] + 2 * c["hidden"], "flops": 12 * c["tokens"] * c["hidden"]}


def tolerance(case):
    """About four times what a pass differs by from the same computation in 64 bits: 2.0e-4 .. 2.8e-4
    (largest single difference 1.2e-3) for the attention calls, whose output is rounded to fp16 once;
    5.1e-4 .. 5.7e-4 (9.8e-3) through a layer or a model, which rounds after every projection; 3.7e-4
    (1.3e-3) for the operators."""
    if case["kind"] in ("layer", "model"):
        return {"rel": 2.2e-3, "max": 0.04}
    return {"rel": 1.5e-3, "max": 6e-3} if case["kind"] == "ops" else {"rel": 1e-3, "max": 5e-3}


# ---- inputs ------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, sigma=1.0):
    return torch.empty(shape, dtype=HALF, device=DEV).normal_(0.0, sigma, generator=g)


def _pool_mb(chunks, c):
    return -(-chunks * c["chunk"] * c["heads"] * D * 4 // (1 << 20)) + 1


def _cache(c, chunks):
    return Attention(c["heads"], D, c["chunk"], memory_mb=_pool_mb(chunks, c), dtype=HALF, device=torch.device(DEV))


def _prompts(c):
    """(token ids, (lengths of the root, group and private parts)) of every sequence."""
    out = []
    for s, n in enumerate(_lengths(c)):
        group = c.get("group", 0)
        g = s // c.get("per_group", 1)
        ids = list(range(c["root"])) + list(range(1_000_000 + 10_000 * g, 1_000_000 + 10_000 * g + group)) + \
            list(range(10_000_000 + 10_000 * s, 10_000_000 + 10_000 * s + n))
        out.append((ids, (c["root"], group, n)))
    return out


def _forward_inputs(c, seed):
    """Every sequence's (token ids, k, v), then the queries.  k and v are views of buffers that the
    next sequence's private tokens overwrite."""
    g, h = _gen(seed), c["heads"]
    prompts = _prompts(c)
    longest = max(len(ids) for ids, _ in prompts)
    k, v = (torch.empty((longest, h, D), dtype=HALF, device=DEV) for _ in range(2))
    root, group = c["root"], c["group"]
    for t in (k, v):
        t[:root].normal_(generator=g)
    for s, (ids, _) in enumerate(prompts):
        for t in (k, v):
            if group and s % c["per_group"] == 0:
                t[root:root + group].normal_(generator=g)
            t[root + group:len(ids)].normal_(generator=g)
        yield ids, k[:len(ids)], v[:len(ids)]
    yield _normal(g, c["batch"], h, D)


def _prepare_forward(c, seed):
    attn = _cache(c, sum(len(ids) // c["chunk"] + 2 for ids, _ in _prompts(c)))
    inputs = _forward_inputs(c, seed)
    for _ in range(c["batch"]):
        attn.add_seq(*next(inputs))
    attn.refresh_kernel_context()
    return {"kind": "forward", "attn": attn, "q": next(inputs)}


def _generate_inputs(c, seed):
    g, h, n = _gen(seed), c["heads"], c["batch"]
    prompts = _prompts(c)
    root_k, root_v = _normal(g, c["root"], h, D), _normal(g, c["root"], h, D)
    requests = []
    for ids, (_, _, own) in prompts:
        requests.append((ids, torch.cat([root_k, _normal(g, own, h, D)]), torch.cat([root_v, _normal(g, own, h, D)])))
    steps = [([20_000_000 + 1000 * t + s for s in range(n)], _normal(g, n, h, D), _normal(g, n, h, D), _normal(g, n, h, D))
             for t in range(c["steps"])]
    return requests, steps


def _prepare_generate(c, seed):
    requests, steps = _generate_inputs(c, seed)
    chunks = sum((len(ids) + c["steps"]) // c["chunk"] + 2 for ids, _, _ in requests)
    return {"kind": "generate", "attn": _cache(c, chunks), "requests": requests, "steps": steps}


def _beam_inputs(c, seed):
    g, h, width = _gen(seed), c["heads"], c["width"]
    prompt = (list(range(c["prompt"])), _normal(g, c["prompt"], h, D), _normal(g, c["prompt"], h, D))
    steps = []
    for t in range(c["steps"]):
        first = t == 0
        # the first step opens the beams; later ones give the beam that leads two candidates and every
        # other one a single one, and drop the beam that is then the last
        counts = [width] if first else [2 if b == (7 * t) % width else 1 for b in range(width)]
        parts = []
        for b, m in enumerate(counts):
            parts.append(([1_000_000 + 1000 * t + 10 * b + i for i in range(m)], _normal(g, m, h, D), _normal(g, m, h, D)))
        steps.append((parts, None if first else (11 * t + 3) % (width + 1), _normal(g, width, h, D)))
    return prompt, steps


def _prepare_beam(c, seed):
    prompt, steps = _beam_inputs(c, seed)
    chunks = c["prompt"] // c["chunk"] + (c["width"] + 2) * (c["steps"] // c["chunk"] + 3)
    return {"kind": "beam", "attn": _cache(c, chunks), "prompt": prompt, "steps": steps}


def _prepare_layer(c, seed):
    g, hidden, batch = _gen(seed), c["heads"] * D, c["batch"]
    layer = LlamaChunkAttention(hidden, c["heads"], device=DEV)
    with torch.no_grad():
        for p in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj):
            p.weight.normal_(0.0, 1.0 / math.sqrt(hidden), generator=g)
    n = c["prompt"]
    seqs = [[10_000 * s + i for i in range(n)] for s in range(batch)]
    positions = torch.arange(n, dtype=torch.int64, device=DEV).repeat(batch, 1)
    steps = []
    for t in range(c["steps"]):
        longer = [seq + [5_000_000 + i for i in range(t + 1)] for seq in seqs]
        steps.append((_normal(g, batch, 1, hidden), longer, torch.full((batch, 1), n + t, dtype=torch.int64, device=DEV)))
    kv = capi.Attention(c["heads"], D, c["chunk"], memory_mb=_pool_mb(batch * ((n + c["steps"]) // c["chunk"] + 2), c),
                        dtype=HALF, device=torch.device(DEV))
    return {"kind": "layer", "layer": layer, "kv": kv, "prompt": (_normal(g, batch, n, hidden), seqs, positions), "steps": steps}


def _prepare_model(c, seed):
    chunks = c["batch"] * ((c["root"] + c["unique"] + c["steps"]) // c["chunk"] + 2)
    model = AttentionOnlyLM(c["vocab"], c["heads"] * D, c["heads"], c["layers"], chunk_size=c["chunk"],
                            memory_mb=_pool_mb(chunks, c), seed=seed, device=DEV)
    draws = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, c["vocab"], (c["root"] + c["batch"] * (c["unique"] + c["steps"]),), generator=draws).tolist()
    root, rest = ids[:c["root"]], ids[c["root"]:]
    each = c["unique"] + c["steps"]
    own = [rest[s * each:(s + 1) * each] for s in range(c["batch"])]
    return {"kind": "model", "model": model, "caches": model.create_kv_caches(),
            "prompts": [root + o[:c["unique"]] for o in own], "answers": [o[c["unique"]:] for o in own], "n_steps": c["steps"]}


def _prepare_ops(c, seed):
    g, n, hidden = _gen(seed), c["tokens"], c["hidden"]
    freqs = torch.arange(4096, device=DEV).float()[:, None] / 10000.0 ** (torch.arange(0, D, 2, device=DEV).float() / D)
    return {"kind": "ops", "x": _normal(g, n, hidden), "residual": _normal(g, n, hidden),
            "weight": 1.0 + _normal(g, hidden, sigma=0.1), "q": _normal(g, n, hidden), "k": _normal(g, n, hidden),
            "cos_sin": torch.cat([freqs.cos(), freqs.sin()], dim=1).to(HALF).contiguous(),
            "positions": torch.arange(n, dtype=torch.int64, device=DEV) % 4096, "neox": c["neox"]}


def prepare(case, seed):
    return {"forward": _prepare_forward, "generate": _prepare_generate, "beam": _prepare_beam, "layer": _prepare_layer,
            "model": _prepare_model, "ops": _prepare_ops}[case["kind"]](case, seed)


# ---- one pass ------------------------------------------------------------------------------------------

def _run_forward(s):
    return s["attn"].forward(s["q"])


def _run_generate(s):
    attn, out = s["attn"], []
    for ids, k, v in s["requests"]:
        attn.add_seq(ids, k, v)
    for tokens, q, k, v in s["steps"]:
        out.append(attn.decode_step(tokens, q, k, v))
    attn.clear()
    return out


def _run_beam(s):
    attn, out = s["attn"], []
    attn.add_seq(*s["prompt"])
    for parts, lost, q in s["steps"]:
        at = 0
        for tokens, k, v in parts:
            attn.append_completion(at, tokens, k, v)
            at += len(tokens)
        if lost is not None:
            attn.remove_seq(lost)
        out.append(attn.forward(q))
    attn.clear()
    return out


@torch.inference_mode()
def _run_layer(s):
    layer, kv = s["layer"], s["kv"]
    out = [layer(*s["prompt"], kv, True)]
    for hidden, seqs, positions in s["steps"]:
        out.append(layer(hidden, seqs, positions, kv, False))
    kv.clear()
    return out


@torch.inference_mode()
def _run_model(s):
    model, caches = s["model"], s["caches"]
    running, answers, out = [], [], []
    for prompt, answer in zip(s["prompts"], s["answers"]):
        seq = Sequence(prompt)
        out.append(model.logits([seq], caches, True))
        running.insert(seq.index, seq)
        answers.insert(seq.index, answer)
    for t in range(s["n_steps"]):
        for seq, answer in zip(running, answers):
            seq.append(answer[t])
        out.append(model.logits(running, caches, False))
    for cache in caches:
        cache.clear()
    return out


def _run_ops(s):
    ops.fused_add_rms_norm(s["x"], s["residual"], s["weight"], 1e-6)
    ops.rotary_embedding(s["positions"], s["q"], s["k"], D, s["cos_sin"], s["neox"])
    return {"x": s["x"], "residual": s["residual"], "q": s["q"], "k": s["k"]}


def run(state):
    return {"forward": _run_forward, "generate": _run_generate, "beam": _run_beam, "layer": _run_layer,
            "model": _run_model, "ops": _run_ops}[state["kind"]](state)


# ---- the same in 64 bits ---------------------------------------------------------------------------------

def _attend(q, k, v):
    """q [h, d], k and v [n, h, d] -> [h, d]."""
    q, k, v = (t.double() for t in (q, k, v))
    p = torch.softmax((k * q).sum(-1) / math.sqrt(D), dim=0)
    return (p[:, :, None] * v).sum(0)


def _exact_forward(c, seed):
    def one(attended):       # the queries come last: two passes over the same draws
        inputs = _forward_inputs(c, seed)
        rows = [attended(s, *next(inputs)[1:]) for s in range(c["batch"])]
        return rows, next(inputs)
    _, q = one(lambda s, k, v: None)
    return torch.stack(one(lambda s, k, v: _attend(q[s], k, v))[0])


def _exact_generate(c, seed):
    requests, steps = _generate_inputs(c, seed)
    out = []
    for s, (_, k, v) in enumerate(requests):
        k = torch.cat([k] + [step[2][s:s + 1] for step in steps])
        v = torch.cat([v] + [step[3][s:s + 1] for step in steps])
        n = k.shape[0] - len(steps)
        out.append(torch.stack([_attend(step[1][s], k[:n + t + 1], v[:n + t + 1]) for t, step in enumerate(steps)]))
    return list(torch.stack(out, dim=1))


def _exact_beam(c, seed):
    (_, k, v), steps = _beam_inputs(c, seed)
    beams, out = [(k, v)], []
    for parts, lost, q in steps:
        grown = []
        for (bk, bv), (tokens, k, v) in zip(beams, parts):
            grown += [(torch.cat([bk, k[i:i + 1]]), torch.cat([bv, v[i:i + 1]])) for i in range(len(tokens))]
        if lost is not None:
            del grown[lost]
        beams = grown
        out.append(torch.stack([_attend(q[b], bk, bv) for b, (bk, bv) in enumerate(beams)]))
    return out


def _rotated(x, positions, table, neox):
    """x [n, heads, d] turned by the angles that `table` has for `positions`."""
    cos, sin = table.double()[positions].chunk(2, dim=-1)
    cos, sin = cos[:, None], sin[:, None]
    if neox:
        a, b = x.chunk(2, dim=-1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], dim=-1).flatten(-2)


def _normed(x, weight, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * weight.double()


def _causal_layer(layer, x):
    """One attention layer over a whole sequence, x [n, hidden]."""
    n, h = x.shape[0], x.shape[1] // D
    q, k, v = ((x @ p.weight.double().t()).view(n, h, D) for p in (layer.q_proj, layer.k_proj, layer.v_proj))
    positions = torch.arange(n, device=x.device)
    q, k = (_rotated(t, positions, layer.rotary_emb.cos_sin_cache, True) for t in (q, k))
    future = torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1)
    heads = [torch.softmax((q[:, i] @ k[:, i].t() / math.sqrt(D)).masked_fill(future, float("-inf")), dim=-1) @ v[:, i]
             for i in range(h)]
    return torch.cat(heads, dim=-1) @ layer.o_proj.weight.double().t()


@torch.no_grad()
def _exact_layer(c, seed):
    s = _prepare_layer(c, seed)
    n, x = c["prompt"], torch.cat([s["prompt"][0]] + [step[0] for step in s["steps"]], dim=1).double()
    whole = torch.stack([_causal_layer(s["layer"], row) for row in x])
    return [whole[:, :n]] + [whole[:, n + t:n + t + 1] for t in range(c["steps"])]


@torch.no_grad()
def _exact_model(c, seed):
    s = _prepare_model(c, seed)
    model, n = s["model"], c["root"] + c["unique"]
    each = []
    for prompt, answer in zip(s["prompts"], s["answers"]):
        x = model.embed_tokens.weight[torch.tensor(prompt + answer, device=DEV)].double()
        for norm, layer in zip(model.input_norms, model.layers):
            x = x + _causal_layer(layer, _normed(x, norm.weight, norm.eps))
        each.append(_normed(x[n - 1:], model.norm.weight, model.norm.eps) @ model.lm_head.weight.double().t())
    return [e[:1] for e in each] + [torch.stack([e[t + 1] for e in each]) for t in range(c["steps"])]


def _exact_ops(c, seed):
    s = _prepare_ops(c, seed)
    residual = s["residual"].double() + s["x"].double()
    q, k = (_rotated(s[t].double().view(c["tokens"], -1, D), s["positions"], s["cos_sin"], c["neox"]).flatten(1) for t in "qk")
    return {"x": _normed(residual, s["weight"], 1e-6), "residual": residual, "q": q, "k": k}


def exact(case, seed):
    return {"forward": _exact_forward, "generate": _exact_generate, "beam": _exact_beam, "layer": _exact_layer,
            "model": _exact_model, "ops": _exact_ops}[case["kind"]](case, seed)
