"""The work that this engine is measured on: whole generations through LLMEngine.generate, and given token ids
fed step by step through TraceReplayer.run_step, which returns the logits.

Sizes are this repository's own: its tiny 32-bit test model, the 50.9M model of bench.py, the GPT-2-small shape and
the width of the GPT-2-XL shape (12 of its layers, which are all alike), and the Bobevik and Viperax models of
`bench.py --compare`.  Prompt lengths of a case are fixed by the case; weights and token ids come from the seed.
"""

import json
import math
import os
import random
import shutil
import tempfile

import numpy as np
import torch

PAGE = 16
TORCH = {"bfloat16": torch.bfloat16, "float32": torch.float32}
BASE = {"arch": "gpt2-mini", "kind": "replay", "dtype": "bfloat16", "layers": 8, "width": 512, "heads": 8, "vocab": 50304,
        "bias": True, "requests": 1, "shortest": 128, "longest": 128, "new": 0, "portion": 0, "rows": "last",
        "table_std": 0.02, "temperature": 0.0, "top_k": 0, "top_p": 1.0}
# A table drawn this wide gives the tied head the sharp distributions of a trained model, so that which token is
# generated does not hang on the rounding of bfloat16.
SHARP = 0.1


def _case(name, **fields):
    return {"name": name, **BASE, **fields}


def listed():
    return [
        # The smallest call: the repository's tiny model in 32 bits, three short prompts; latency and launches.
        _case("tiny_f32_generate", kind="generate", dtype="float32", layers=2, width=64, heads=4, vocab=257, requests=3,
              shortest=5, longest=30, new=12),
        # One user of the 50.9M model: a prompt of 128 tokens, 64 greedy ones; the latency of a decode step.
        _case("50m_generate_b1", kind="generate", table_std=SHARP, new=64),
        # The headline of bench.py: eight requests decoded together.
        _case("50m_generate_b8", kind="generate", table_std=SHARP, requests=8, new=64),
        # A busy server of the 50.9M model: 64 requests, sampled with temperature, top-k and top-p.
        _case("50m_generate_b64_sampled", kind="generate", table_std=SHARP, requests=64, new=32, temperature=0.8, top_k=50,
              top_p=0.95),
        # Prefill as bench.py measures it: two prompts of 1,024 tokens in one step.
        _case("50m_prefill_2048", requests=2, shortest=1024, longest=1024),
        # Continuous batching on the GPT-2-small shape: prompts of any length arrive one after another and are cut into
        # portions of at most 512 tokens, each beside a decoded token of every request that is through its prompt.
        _case("small_mixed", layers=12, width=768, heads=12, vocab=50257, requests=12, shortest=16, longest=960, portion=512,
              new=4),
        # Long prompts at the width of the XL shape: large products, attention over 1,024 keys.
        _case("wide_prefill_4096", layers=12, width=1600, heads=25, vocab=50257, requests=4, shortest=1024, longest=1024),
        # A batch of 32 ragged requests at that width: a prompt step, then decode steps that read all weights.
        _case("wide_decode_b32", layers=12, width=1600, heads=25, vocab=50257, requests=32, shortest=40, longest=240, new=16),
        # The true 32-bit path over ragged prompts, as a checking run scores them: logits at every token.
        _case("50m_f32_score", dtype="float32", requests=4, shortest=1, longest=640, rows="all"),
        # The true 32-bit path of the GPT-2-small shape end to end: ragged prompts, sampled tokens.
        _case("small_f32_generate", kind="generate", dtype="float32", layers=12, width=768, heads=12, vocab=50257, requests=16,
              shortest=16, longest=256, new=24, temperature=0.8, top_k=50, top_p=0.95),
        # Softmax attention mixed with a decaying state, gated feed-forwards: ragged prompts, then decode steps.
        _case("bobevik_prompts_and_decode", arch="Bobevik", layers=4, width=1024, heads=8, vocab=32768, requests=8, shortest=100,
              longest=1024, new=16),
        # Latent attention behind a window, experts chosen by a table, several residual streams: prompts, then decode steps.
        _case("viperax_prompts_and_decode", arch="Viperax", layers=4, width=2048, heads=16, vocab=32768, requests=8, shortest=64,
              longest=700, new=16),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _cost(case):
    """Roughly the seconds of a pass: matrix work at the rate of the type, bytes, and steps of dependent kernels."""
    w = work(case)
    return (w["flops"] / (4e14 if case["dtype"] == "bfloat16" else 1e13) + w["bytes"] / 4e12
            + len(_steps(case)) * (case["layers"] + 2) * 2e-5)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        arch = rng.choice(["gpt2-mini"] * 6 + ["Bobevik", "Viperax"])
        case = dict(BASE, arch=arch, dtype=rng.choice(["bfloat16", "bfloat16", "float32"]))
        if arch == "gpt2-mini":
            head = rng.choice([16, 32]) if rng.random() < 0.2 else 64
            heads = _log_int(rng, 1 if head < 64 else 4, 8 if head < 64 else 25)
            case.update(kind=rng.choice(["replay", "replay", "generate"]), layers=_log_int(rng, 2, 12), heads=heads,
                        width=heads * head, bias=rng.random() < 0.7,
                        vocab=rng.choice([50304, 50257, _log_int(rng, 257, 60000)]))
        else:
            case.update(dtype="bfloat16", layers=rng.choice([2, 4]), vocab=32768)
            case.update(heads=rng.choice([8, 16]))
            case.update(width=128 * case["heads"])
        case.update(requests=_log_int(rng, 1, 64), shortest=_log_int(rng, 1, 256))
        case.update(longest=max(case["shortest"], _log_int(rng, 8, 960)), new=rng.choice([0, _log_int(rng, 4, 48)]))
        if case["kind"] == "generate":
            case.update(new=max(case["new"], 4), table_std=SHARP if case["dtype"] == "bfloat16" else 0.02)
            if rng.random() < 0.5:
                case.update(temperature=round(rng.uniform(0.5, 1.2), 2), top_k=rng.choice([0, 20, 50]),
                            top_p=rng.choice([1.0, 0.9, 0.95]))
        elif case["new"]:
            case.update(portion=rng.choice([0, 0, 256, 512]))
        elif sum(_lengths(case)) * case["vocab"] <= 6e7:
            case.update(rows=rng.choice(["last", "all"]))
        ends = max(before + q for step in _steps(case) for _, before, q in step)
        if ends <= 1024 and sum(_lengths(case)) <= 16384 and _cost(case) <= most:
            return case


# ---------------------------------------------------------------- what a case asks of the engine
def _lengths(case):
    """Prompt lengths: spread between the case's ends, both of them among them, in a shuffled order."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    rng = random.Random(json.dumps([n, lo, hi]))
    lengths = [lo, hi][:n] + [rng.randint(lo, hi) for _ in range(n - 2)]
    rng.shuffle(lengths)
    return lengths


def _tokens(case, seed):
    """Per request the prompt's ids and, for a replay, the ids that follow it."""
    rng = np.random.default_rng([seed, 7])
    taken = [0] * case["requests"]
    for step in _steps(case):
        for r, _, q in step:
            taken[r] += q
    return [rng.integers(0, case["vocab"], n).tolist() for n in taken]


def _steps(case):
    """[[(request, tokens before, tokens in this step)]]: the prompts in one step and then one token of each at a time;
    or, with portions, the prompts one after another beside single tokens of the requests whose prompt is through.
    In a generation the prompt's step makes the first of the new tokens."""
    lengths, steps = _lengths(case), []
    done = [0] * len(lengths)
    if case["portion"]:
        for i, n in enumerate(lengths):
            while done[i] < n:
                step = [(r, done[r], 1) for r in range(i)] + [(i, done[i], min(case["portion"], n - done[i]))]
                steps.append(step)
                for r, _, q in step:
                    done[r] += q
    else:
        steps.append([(i, 0, n) for i, n in enumerate(lengths)])
        done = list(lengths)
    for _ in range(case["new"] - (case["kind"] == "generate")):
        steps.append([(r, done[r], 1) for r in range(len(done))])
        done = [d + 1 for d in done]
    return steps


def _wanted(case, step):
    """[(request, tokens up to the row)] whose logits are asked for: every token's, or the last one's of each request that
    is not in the middle of its prompt."""
    if case["rows"] == "all":
        return [(r, before + t + 1) for r, before, q in step for t in range(q)]
    lengths = _lengths(case)
    return [(r, before + q) for r, before, q in step if before + q >= lengths[r]]


# ---------------------------------------------------------------- models: config.json and tensors
def _config(case):
    layers, width, heads, vocab = case["layers"], case["width"], case["heads"], case["vocab"]
    if case["arch"] == "gpt2-mini":
        return {"architecture": "gpt2-mini", "n_layer": layers, "n_embd": width, "n_head": heads, "vocab_size": vocab,
                "block_size": 1024, "bias": case["bias"], "layer_norm_eps": 1e-5}
    out = []
    for i in range(layers):
        if case["arch"] == "Bobevik":
            kind = ["parallel", "retention", "attention", "retention"][i % 4] if layers > 2 else ["parallel", "attention"][i]
            half, state = max(heads // 2, 1), {"heads": heads, "dim": 128, "vdim": 128}
            mixer = {
                "retention": {**state, "decay": [1.0 - 2.0 ** (-5 - h % 8) for h in range(heads)], "rot": {"dims": 64, "base": 1e6}},
                "attention": {**state, "kv_heads": heads // 4, "scale": 128 ** -0.5, "rot": {"dims": 128, "base": 10000.0},
                              "v_mix": True},
                "parallel": {"left": {**state, "heads": half, "kv_heads": max(half // 4, 1), "scale": 128 ** -0.5,
                                      "rot": {"dims": 64, "base": 50000.0, "scaling": {"factor": 4.0}}, "softcap": 30.0},
                             "right": {**state, "heads": half, "decay": [1.0 - 2.0 ** (-1 - h % 10) for h in range(half)]}},
            }[kind]
            out.append({"type": kind, "mixer": mixer, "mlp": {"kind": "dense", "ff": width * 8 // 3 // 64 * 64}})
        else:
            mixer = {"heads": heads, "dim": 128, "vdim": 128, "kv_rank": 128, "scale": 128 ** -0.5, "mask": {"size": 512}}
            if layers >= 4 and i >= layers // 2:
                mixer["kv_from"] = layers // 2 - 1
            mlp = ({"kind": "moe", "expert": {"ff": width}, "router": {"experts": 8, "top": 2},
                    "shared": {"ff": width * 2 // 3 // 64 * 64}} if i % 2
                   else {"kind": "dense", "ff": width * 8 // 3 // 64 * 64})
            out.append({"type": "latent_attention", "mixer": mixer, "mlp": mlp})
    raw = {"architecture": case["arch"], "vocab": vocab, "width": width, "norm": {"eps": 1e-5}, "layers": out}
    if case["arch"] == "Bobevik":
        return {**raw, "residual_mult": 0.7}
    return {**raw, "streams": 2, "embedding": {"scale": float(width) ** 0.5}, "logit_scale": 1.0, "logit_softcap": 30.0}


def _shapes(case):
    """[(tensor, shape, mean, standard deviation)]; a mean of "distinct" stands for rows of different expert numbers."""
    cfg, c, vocab = _config(case), case["width"], case["vocab"]
    if case["arch"] == "gpt2-mini":
        std, res = 0.02, 0.02 / math.sqrt(2 * case["layers"])
        plan = [("tok_emb.weight", (vocab, c), 0.0, case["table_std"]), ("pos_emb.weight", (cfg["block_size"], c), 0.0, std)]
        for i in range(case["layers"]):
            p = f"blocks.{i}."
            for name, out, inn, s in (("attn.qkv", 3 * c, c, std), ("attn.proj", c, c, res), ("mlp.fc", 4 * c, c, std),
                                      ("mlp.proj", c, 4 * c, res)):
                plan += [(p + name + ".weight", (out, inn), 0.0, s), (p + name + ".bias", (out,), 0.0, 0.01)]
            for name in ("ln1", "ln2"):
                plan += [(p + name + ".weight", (c,), 1.0, 0.1), (p + name + ".bias", (c,), 0.0, 0.01)]
        plan += [("ln_f.weight", (c,), 1.0, 0.1), ("ln_f.bias", (c,), 0.0, 0.01)]
        return [t for t in plan if case["bias"] or not t[0].endswith(".bias")]
    plan = []

    def lin(name, out, inn):
        plan.append((name, (out, inn), 0.0, inn ** -0.5))

    def gated(p, ff):
        lin(p + "gate", ff, c), lin(p + "up", ff, c), lin(p + "down", c, ff)

    def state(p, m):
        for n, dim in (("q", "dim"), ("k", "dim"), ("v", "vdim"), ("g", "vdim")):
            lin(p + n, m["heads"] * m[dim], c)
        lin(p + "o", c, m["heads"] * m["vdim"])

    def attention(p, m, biases):
        for n, out in (("q", m["heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"]), ("v", m["kv_heads"] * m["vdim"])):
            lin(p + n, out, c)
            if biases:
                plan.append((p + n + ".b", (out,), 0.0, 0.5))
        if m.get("v_mix"):
            plan.append((p + "vmix", (), 0.4, 0.25))
        lin(p + "g", m["heads"], c)
        lin(p + "o", c, m["heads"] * m["vdim"])

    bob = case["arch"] == "Bobevik"
    plan.append(("embed", (vocab, c), 0.0, 1.0 if bob else c ** -0.5))
    if bob:
        plan.append(("embed.norm", (c,), 0.0, 0.1))
    for i, layer in enumerate(cfg["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        plan += [(p + n, (c,), 0.0 if bob else 1.0, 0.1) for n in (("norm1", "norm1b", "norm2", "norm2b") if bob else
                                                                   ("norm1", "norm2"))]
        if layer["type"] == "retention":
            state(p + "mix.", m)
        elif layer["type"] == "attention":
            attention(p + "mix.", m, False)
        elif layer["type"] == "parallel":
            attention(p + "mix.left.", m["left"], True)
            state(p + "mix.right.", m["right"])
            plan += [(p + "mix.right.norm", (m["right"]["heads"] * 128,), 1.0, 0.1)]
            plan += [(p + f"mix.{side}.out", (c,), 1.0, 0.1) for side in ("left", "right")]
        else:
            lin(p + "mix.q", m["heads"] * 128, c)
            if "kv_from" not in m:
                lin(p + "mix.dkv", 128, c)
                plan.append((p + "mix.dkv.norm", (128,), 1.0, 0.1))
            lin(p + "mix.uk", m["heads"] * 128, 128), lin(p + "mix.uv", m["heads"] * 128, 128)
            plan.append((p + "mix.sink", (m["heads"],), 0.0, 1.0))
            lin(p + "mix.g", m["heads"] * 128, c), lin(p + "mix.o", c, m["heads"] * 128)
            for h in "12":
                plan += [(f"{p}hc{h}.in", (2,), 0.5, 0.25), (f"{p}hc{h}.out", (2,), 1.0, 0.2),
                         (f"{p}hc{h}.mix", (2, 2), "identity", 0.1)]
        if f["kind"] == "dense":
            gated(p + "mlp.", f["ff"])
        else:
            for e in range(8):
                gated(f"{p}mlp.e{e}.", f["expert"]["ff"])
            gated(p + "mlp.shared.", f["shared"]["ff"])
            plan.append((p + "mlp.table", (vocab, 2), "distinct", 8))
    plan.append(("final.norm", (c,), 0.0 if bob else 1.0, 0.1))
    lin("head", vocab, c)
    return plan


def _weights(case, seed):
    """Tensors by name in the type that the model folder stores, on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * seed + 17)
    out = {}
    for name, shape, mean, std in _shapes(case):
        if mean == "distinct":
            out[name] = torch.rand((shape[0], std), generator=gen, device="cuda").argsort(dim=1)[:, :shape[1]].to(torch.int32)
            continue
        t = torch.empty(shape, device="cuda").normal_(0.0, std, generator=gen)
        t += torch.eye(shape[0], device="cuda") if mean == "identity" else mean
        out[name] = t.to(TORCH[case["dtype"]])
    return out


def _write_folder(path, case, seed):
    """config.json and model.safetensors (the header's length, the header, the tensors one behind the other)."""
    with open(os.path.join(path, "config.json"), "w", encoding="utf-8") as fh:
        json.dump(_config(case), fh)
    tensors = {k: v.contiguous().cpu() for k, v in _weights(case, seed).items()}
    names = {torch.bfloat16: "BF16", torch.float32: "F32", torch.int32: "I32"}
    header, at = {}, 0
    for k, t in tensors.items():
        size = t.numel() * t.element_size()
        header[k] = {"dtype": names[t.dtype], "shape": list(t.shape), "data_offsets": [at, at + size]}
        at += size
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "model.safetensors"), "wb") as fh:
        fh.write(len(text).to_bytes(8, "little") + text)
        for t in tensors.values():
            fh.write(t.reshape(-1).view(torch.uint8).numpy().data)


# ---------------------------------------------------------------- the measured interface
def prepare(case, seed):
    from mini_gpt_inference_amd import EngineConfig, LLMEngine, SamplingParams
    from mini_gpt_inference_amd.engine.replay import TraceReplayer

    tokens, lengths, n = _tokens(case, seed), _lengths(case), case["requests"]
    folder = tempfile.mkdtemp(prefix="cases_")
    try:
        _write_folder(folder, case, seed)
        if case["kind"] == "generate":
            pages = sum(-(-(length + case["new"]) // PAGE) for length in lengths)
            engine = LLMEngine.from_folder(folder, EngineConfig(
                block_size=PAGE, num_blocks=max(pages + 8, 64), max_batch_size=max(n, 2),
                max_num_batched_tokens=max(4096, sum(lengths)), dtype=case["dtype"]))
            engine.capture_decode_graphs([n])
            params = [SamplingParams(max_tokens=case["new"], temperature=case["temperature"], top_k=case["top_k"] or None,
                                     top_p=case["top_p"] if case["top_p"] < 1.0 else None, seed=seed + i) for i in range(n)]
            return {"engine": engine, "prompts": [t[:length] for t, length in zip(tokens, lengths)], "params": params}
        rooms = sum(-(-len(t) // PAGE) * PAGE for t in tokens)
        replayer = TraceReplayer(folder, case["dtype"], rooms, max_live=n)
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    records = []
    for s, step in enumerate(_steps(case)):
        wanted = _wanted(case, step)
        records.append({"step": s, "entries": [{"id": f"r{r}", "tokens": tokens[r][before:before + q],
                                                "want": [end - before - 1 for who, end in wanted if who == r]}
                                               for r, before, q in step]})
    records[-1]["end"] = [f"r{r}" for r in range(n)]
    return {"replayer": replayer, "records": records}


def run(state):
    if "engine" in state:
        return {"tokens": np.array(state["engine"].generate(state["prompts"], state["params"]), dtype=np.int64)}
    # a step's logits lie in the replayer's workspace until the next step: a caller keeps copies
    logits = []
    for record in state["records"]:
        step = state["replayer"].run_step(record)
        if step is not None:
            logits.append(step.clone())
    return logits


def work(case):
    """Per step: every matrix that its tokens go through once, the cached keys, values and states that they read, the logits
    that come back (in a generation, the tokens); multiply-adds of the matrices and of attention over the keys seen."""
    size = 2 if case["dtype"] == "bfloat16" else 4
    cfg, c, vocab = _config(case), case["width"], case["vocab"]
    always = top = expert = 0                      # elements a token goes through; of the experts: chosen, and of one
    for name, shape, *_ in _shapes(case):
        if len(shape) == 2 and name not in ("tok_emb.weight", "pos_emb.weight", "embed", "head") and not name.endswith(".table"):
            if ".mlp.e" in name:
                top += shape[0] * shape[1] * 2 // 8
                expert += shape[0] * shape[1] // 8
            else:
                always += shape[0] * shape[1]
    attending = []                                 # per layer: (query heads x head size, cached values a token, window)
    state = 0
    for i in range(case["layers"]):
        if case["arch"] == "gpt2-mini":
            attending.append((c, 2 * c, 0))
            continue
        kind, m = cfg["layers"][i]["type"], cfg["layers"][i]["mixer"]
        if kind == "latent_attention":
            attending.append((m["heads"] * 128, 128, 512))
        for a in [m] if kind == "attention" else [m["left"]] if kind == "parallel" else []:
            attending.append((a["heads"] * 128, 2 * a["kv_heads"] * 128, 0))
        for s in [m] if kind == "retention" else [m["right"]] if kind == "parallel" else []:
            state += s["heads"] * 128 * 128
    moved = flops = 0
    for step in _steps(case):
        n, rows = sum(q for *_, q in step), len(_wanted(case, step))
        flops += 2 * n * (always + top) + 2 * rows * vocab * c + 4 * n * state
        moved += size * (always + expert * min(8, 2 * n) + (vocab * c if rows else 0) + n * c)
        moved += 2 * 4 * state * len(step) + (4 * rows * (1 if case["kind"] == "generate" else vocab))
        for wide, cached, window in attending:
            for _, before, q in step:
                reach = min(before, window) if window else before
                seen = sum(min(before + t + 1, window) for t in range(q)) if window else q * before + q * (q + 1) // 2
                flops += 4 * wide * seen
                moved += size * cached * (reach + q)
    return {"bytes": int(moved), "flops": int(flops)}


def tolerance(case):
    if case["kind"] == "generate":
        return {"rel": 0.0, "differ": 0.005}       # whole tokens
    # Against 64 bits the logits were off by 0.0015 to 0.0073 in bfloat16 (by model), by 1.3e-6 in 32 bits.
    return {"rel": 2e-2, "max": 0.15} if case["dtype"] == "bfloat16" else {"rel": 6e-6, "max": 6e-5}


# ---------------------------------------------------------------- the same in 64 bits
def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _layer_norm(x, gain, bias, eps):
    y = _unit(x - x.mean(dim=-1, keepdim=True), eps) * gain
    return y if bias is None else y + bias


def _attend(q, k, v, scale, softcap=0.0, window=0, sink=None):
    """q [T, H, D], k and v [T, G, .] -> [T, H, .]: causal softmax attention, a score more per head with a sink."""
    heads, t = q.shape[1], torch.arange(q.shape[0], device=q.device)
    back = t[:, None] - t[None, :]
    hidden = (back < 0) | (back >= (window or len(t)))
    out = []
    for h in range(heads):
        g = h * k.shape[1] // heads
        s = (q[:, h] @ k[:, g].T) * scale
        s = (softcap * torch.tanh(s / softcap) if softcap else s).masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(len(t), 1)], dim=1)
        out.append(torch.softmax(s, dim=-1)[:, :len(t)] @ v[:, g])
    return torch.stack(out, dim=1)


def _rotate(x, rot):
    if not rot:
        return x
    dims, half = rot["dims"], rot["dims"] // 2
    freq = rot["base"] ** (-2.0 * torch.arange(half, device=x.device, dtype=x.dtype) / dims)
    angle = torch.arange(len(x), device=x.device, dtype=x.dtype)[:, None] * freq / rot.get("scaling", {}).get("factor", 1.0)
    cos, sin, a, b = torch.cos(angle)[:, None], torch.sin(angle)[:, None], x[..., :half], x[..., half:dims]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., dims:]], dim=-1)


def _gpt(w, cfg, ids):
    eps, heads = cfg["layer_norm_eps"], cfg["n_head"]
    x = w["tok_emb.weight"][ids] + w["pos_emb.weight"][:len(ids)]
    norm = lambda x, p: _layer_norm(x, w[p + ".weight"], w.get(p + ".bias"), eps)
    lin = lambda x, p: x @ w[p + ".weight"].T + w.get(p + ".bias", 0.0)
    for i in range(cfg["n_layer"]):
        p = f"blocks.{i}."
        q, k, v = lin(norm(x, p + "ln1"), p + "attn.qkv").view(len(ids), 3, heads, -1).unbind(1)
        x = x + lin(_attend(q, k, v, q.shape[-1] ** -0.5).flatten(1), p + "attn.proj")
        u = lin(norm(x, p + "ln2"), p + "mlp.fc")
        x = x + lin(torch.nn.functional.gelu(u, approximate="tanh"), p + "mlp.proj")
    return norm(x, "ln_f"), w["tok_emb.weight"]


def _decay(q, k, v, decay):
    """Per head S <- decay S + k v^T and S^T q, as a product with the decays between tokens."""
    t = torch.arange(len(q), device=q.device, dtype=q.dtype)
    back = t[:, None] - t[None, :]
    out = []
    for h, d in enumerate(decay):
        between = torch.where(back >= 0, d ** back.clamp(min=0), torch.zeros_like(back))
        out.append(((q[:, h] @ k[:, h].T) * between) @ v[:, h])
    return torch.stack(out, dim=1)


def _bobevik(w, cfg, ids):
    eps, act = cfg["norm"]["eps"], torch.nn.functional.silu
    norm = lambda x, p: _unit(x, eps) * (1.0 + w[p])

    def state(h, m, p, retention):
        q, k, v = ((h @ w[p + n].T).view(len(ids), m["heads"], -1) for n in "qkv")
        if retention:
            q, k = _rotate(q, m["rot"]), _rotate(k, m["rot"]) * m["dim"] ** -0.5
            o = _unit(_decay(q, k, v, m["decay"]), eps).flatten(1) * act(h @ w[p + "g"].T)
        else:
            o = _unit(_decay(act(q), act(k), act(v), m["decay"]).flatten(1), eps) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].T)
        return o @ w[p + "o"].T

    def attention(h, m, p, biases):
        bias = (lambda n: w[p + n + ".b"]) if biases else (lambda n: 0.0)
        q, k, v = ((h @ w[p + n].T + bias(n)).view(len(ids), -1, m["dim"]) for n in "qkv")
        q, k = _rotate(q, m.get("rot")), _rotate(k, m.get("rot"))
        if not biases:
            q, k = _unit(q, eps), _unit(k, eps)
        if m.get("v_mix"):
            first = kept.setdefault("values", v)
            v = v if first is v else (1.0 - w[p + "vmix"]) * v + w[p + "vmix"] * first
        o = _attend(q, k, v, m["scale"], m.get("softcap", 0.0)) * torch.sigmoid(h @ w[p + "g"].T)[..., None]
        return o.flatten(1) @ w[p + "o"].T

    kept, x = {}, norm(w["embed"][ids], "embed.norm")
    for i, layer in enumerate(cfg["layers"]):
        p, m, h = f"l{i}.", layer["mixer"], norm(x, f"l{i}.norm1")
        if layer["type"] == "retention":
            y = state(h, m, p + "mix.", True)
        elif layer["type"] == "attention":
            y = attention(h, m, p + "mix.", False)
        else:
            y = 0.5 * (_unit(attention(h, m["left"], p + "mix.left.", True), eps) * w[p + "mix.left.out"]
                       + _unit(state(h, m["right"], p + "mix.right.", False), eps) * w[p + "mix.right.out"])
        x = x + cfg["residual_mult"] * norm(y, p + "norm1b")
        h = norm(x, p + "norm2")
        y = (torch.relu(h @ w[p + "mlp.gate"].T) * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T
        x = x + cfg["residual_mult"] * norm(y, p + "norm2b")
    return norm(x, "final.norm"), w["head"]


def _viperax(w, cfg, ids):
    eps = cfg["norm"]["eps"]
    gated = lambda h, p: (torch.nn.functional.silu(h @ w[p + "gate"].T) * (h @ w[p + "up"].T)) @ w[p + "down"].T

    def mixer(h, i, m, p):
        if "kv_from" not in m:
            kept[i] = _unit(h @ w[p + "dkv"].T, eps) * w[p + "dkv.norm"]
        c = kept[m.get("kv_from", i)]
        q, k, v = ((a @ w[p + n].T).view(len(ids), m["heads"], -1) for a, n in ((h, "q"), (c, "uk"), (c, "uv")))
        o = _attend(q, k, v, m["scale"], window=m["mask"]["size"], sink=w[p + "sink"]).flatten(1)
        return (o * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T

    def feed_forward(h, mlp, p):
        if mlp["kind"] == "dense":
            return gated(h, p)
        y, rows = gated(h, p + "shared."), w[p + "table"].long()[ids]
        for e in range(8):
            mine = (rows == e).any(dim=1).nonzero().flatten()
            y[mine] += gated(h[mine], f"{p}e{e}.") / 2
        return y

    kept, streams = {}, (w["embed"][ids] * cfg["embedding"]["scale"])[None].repeat(cfg["streams"], 1, 1)
    for i, layer in enumerate(cfg["layers"]):
        for n, sub in (("1", lambda h: mixer(h, i, layer["mixer"], f"l{i}.mix.")),
                       ("2", lambda h: feed_forward(h, layer["mlp"], f"l{i}.mlp."))):
            read = (streams * w[f"l{i}.hc{n}.in"][:, None, None]).sum(dim=0)
            y = sub(_layer_norm(read, w[f"l{i}.norm{n}"], None, eps))
            mix = w[f"l{i}.hc{n}.mix"]
            streams = torch.stack([(streams * mix[:, t, None, None]).sum(dim=0) + w[f"l{i}.hc{n}.out"][t] * y
                                   for t in range(cfg["streams"])])
    return _layer_norm(streams.sum(dim=0), w["final.norm"], None, eps), w["head"]


def exact(case, seed):
    """The logits of a replay, every request on its own and its tokens all at once.  Tokens have no 64-bit value."""
    if case["kind"] == "generate":
        return None
    cfg = _config(case)
    w = {k: v.to(torch.float64) for k, v in _weights(case, seed).items()}
    model = {"gpt2-mini": _gpt, "Bobevik": _bobevik, "Viperax": _viperax}[case["arch"]]
    tokens = _tokens(case, seed)
    rows = {}                                      # (request, tokens so far) -> logits
    wanted = [_wanted(case, step) for step in _steps(case)]
    for r, ids in enumerate(tokens):
        hidden, head = model(w, cfg, torch.tensor(ids, device="cuda"))
        ends = sorted({end for step in wanted for q, end in step if q == r})
        logits = hidden[[end - 1 for end in ends]] @ head.T * cfg.get("logit_scale", 1.0)
        if cfg.get("logit_softcap"):
            logits = cfg["logit_softcap"] * torch.tanh(logits / cfg["logit_softcap"])
        rows.update({(r, end): logits[j] for j, end in enumerate(ends)})
    return [torch.stack([rows[key] for key in step]) for step in wanted if step]
