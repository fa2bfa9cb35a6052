"""What is measured: the steps that a program that serves with this framework has it run.

A case is a model of given layer sizes and a pass over it: some requests whose keys (and states) are cached already
decode a few tokens each, or new prompts arrive in portions, or both share the steps.  Everything goes through
`ModelRunner` (captured programs, as `Engine` runs it by default): the decoding requests of a pass are forks of the
cached ones, so that a pass leaves the cache as it found it.  The tokens fed are given ones and not the picked ones (as
when a continuation is scored or forced), because two correct runs part for good after one near-tie; a token is picked
from every row of logits all the same, and read on the host one step later, as the scheduler's overlapped ticks do.

Weights are random with the spread of trained ones (every projection keeps its input's scale, queries and keys are wide
enough for attention that is not uniform, routers are sharp), the same tensors for the framework and for `exact`.
"""
import math
import random
from types import SimpleNamespace

import numpy as np
import torch

GPU = "cuda:0"
PAGE = 16

# -- the models -------------------------------------------------------------------------------------------------------

# layers, width, heads, key/value heads, head size, feed-forward, vocabulary, rotary base, tied head
LLAMA = {
    "smollm2-135m": (30, 576, 9, 3, 64, 1536, 49152, 100000.0, True),
    "smollm2-1.7b": (24, 2048, 32, 32, 64, 8192, 49152, 130000.0, True),
    "llama-3-8b": (32, 4096, 32, 8, 128, 14336, 128256, 500000.0, False),
}


def config_of(case):
    """The config.json of the case's model."""
    name, layers, context = case["model"], case["layers"], 16384
    if name in LLAMA:
        _, width, heads, kv, dim, ff, vocab, theta, tied = LLAMA[name]
        return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_act": "silu", "vocab_size": vocab,
                "hidden_size": width, "intermediate_size": ff, "num_hidden_layers": layers, "num_attention_heads": heads,
                "num_key_value_heads": kv, "head_dim": dim, "rms_norm_eps": 1e-5, "rope_theta": theta,
                "max_position_embeddings": context, "tie_word_embeddings": tied}
    design, width = name.split("-")
    width = int(width)
    heads, kv, ff = width // 128, max(1, width // 512), 4 * width
    base = {"vocab": 32768, "width": width, "norm": {"eps": 1e-5}, "max_positions": context}
    if design == "novosun":      # softmax attention beside a state-space layer, then gated linear attention, in turn
        mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
        order = [{"type": "parallel", "mlp": mlp, "mixer": {
                      "left": {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 128, "scale": 0.125},
                      "right": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}},
                 {"type": "gla", "mlp": mlp, "mixer": {"heads": width // 256, "dim": 128, "vdim": 256, "tau": 16.0}}]
        return {"architecture": "Novosun", "residual_mult": 0.5, "layers": [order[i % 2] for i in range(layers)], **base}
    if design == "ditazen":      # latent attention over all keys, the delta rule, latent attention over a window, the rule
        mlp = {"kind": "dense", "ff": ff}
        latent = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5}
        rule = {"type": "delta", "mlp": mlp, "mixer": {"heads": 2 * heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4}}
        order = [{"type": "latent_attention_2", "mlp": mlp, "mixer": {**latent, "q_rank": 3 * width // 4, "rot": {
                      "base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}, rule,
                 {"type": "latent_attention", "mlp": mlp, "mixer": {**latent, "rot": {"base": 10000.0, "dims": 64}, "mask": {"size": 1024}}}, rule]
        return {"architecture": "Ditazen", "logit_scale": 1.0, "layers": [order[i % 4] for i in range(layers)], **base}
    # noresun: attention with sigmoid weights over a window, the minimal gated unit, attention on the first layer's keys; experts
    mlp = {"kind": "moe", "expert": {"ff": 2 * width}, "router": {"experts": 16, "top": 2}}
    near = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1024},
            "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    unit = {"type": "mingru", "mixer": {"width": width}, "mlp": mlp}
    order = [{"type": "attention", "mixer": near, "mlp": mlp}, unit, {"type": "attention", "mixer": {**near, "kv_from": 0}, "mlp": mlp}, unit]
    return {"architecture": "Noresun", "postln_alpha": 2.0, "layers": [order[i % 4] for i in range(layers)],
            "embedding": {"scale": 1.0, "bigram": {"buckets": 65521, "mul_prev": 131, "mul_cur": 17}}, **base}


def tensors_of(c):
    """{name: (shape, how it is drawn)} of the model: "in" keeps the scale of its input, "out" is added to the residual
    stream, "sharp" is wider (queries and keys, whose scores then spread by 1.4); a number is a spread around zero; "norm", "decay", "step" as named."""
    t = {}
    if "hidden_size" in c:
        W, F, V = c["hidden_size"], c["intermediate_size"], c["vocab_size"]
        q, kv = c["num_attention_heads"] * c["head_dim"], c["num_key_value_heads"] * c["head_dim"]
        t["model.embed_tokens.weight"] = (V, W), 1.0 / math.sqrt(W) * 2.0
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            t[p + "input_layernorm.weight"] = t[p + "post_attention_layernorm.weight"] = (W,), "norm"
            t[p + "self_attn.q_proj.weight"], t[p + "self_attn.k_proj.weight"] = ((q, W), "sharp"), ((kv, W), "sharp")
            t[p + "self_attn.v_proj.weight"], t[p + "self_attn.o_proj.weight"] = ((kv, W), "in"), ((W, q), "out")
            t[p + "mlp.gate_proj.weight"] = t[p + "mlp.up_proj.weight"] = (F, W), "in"
            t[p + "mlp.down_proj.weight"] = (W, F), "out"
        t["model.norm.weight"] = (W,), "norm"
        if not c["tie_word_embeddings"]:
            t["lm_head.weight"] = (V, W), "sharp"
        return t
    W, V = c["width"], c["vocab"]
    t["embed"] = (V, W), (0.5 if c["architecture"] == "Noresun" else 1.0 / math.sqrt(W) * 2.0)
    if c["architecture"] == "Noresun":
        t["bigram"] = (c["embedding"]["bigram"]["buckets"] + 1, W), 0.5
    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
        t[f"l{i}.norm1"] = t[f"l{i}.norm2"] = (W,), "norm"
        kind = layer["type"]
        if kind == "parallel":
            a, s = m["left"], m["right"]
            inner, groups = s["heads"] * s["vdim"], s["groups"] * s["state"]
            t[p + "left.q"], t[p + "left.k"] = ((a["heads"] * a["dim"], W), "in"), ((a["kv_heads"] * a["dim"], W), "in")
            t[p + "left.v"], t[p + "left.o"] = ((a["kv_heads"] * a["vdim"], W), "in"), ((W, a["heads"] * a["vdim"]), "in")
            t[p + "left.g"] = (a["heads"], W), "in"
            t[p + "left.q.norm"] = t[p + "left.k.norm"] = (a["dim"],), "norm"
            t[p + "right.in"], t[p + "right.o"] = ((2 * inner + 2 * groups + s["heads"], W), "in"), ((W, inner), "in")
            t[p + "right.conv"], t[p + "right.conv.b"] = ((inner + 2 * groups, s["conv"]), 0.5), ((inner + 2 * groups,), 0.02)
            t[p + "right.dt_bias"], t[p + "right.A_log"], t[p + "right.D"] = ((s["heads"],), "step"), ((s["heads"],), "decay"), ((s["heads"],), "norm")
            t[p + "right.norm"] = (inner,), "norm"
            t[p + "left.out"] = t[p + "right.out"] = (W,), "norm"
        elif kind == "gla":
            D, E = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            t[p + "q"] = t[p + "k"] = (D, W), "in"
            t[p + "v"] = t[p + "g"] = (E, W), "in"
            t[p + "o"], t[p + "norm"] = ((W, E), "in"), ((m["vdim"],), "norm")
            t[p + "a1"], t[p + "a2"], t[p + "a2.b"] = ((16, W), "in"), ((D, 16), "in"), ((D,), 1.0)
        elif kind.startswith("latent"):
            H, r = m["heads"], m["kv_rank"]
            if "q_rank" in m:
                t[p + "dq"], t[p + "dq.norm"] = ((m["q_rank"], W), "in"), ((m["q_rank"],), "norm")
                t[p + "uq"] = (H * (m["dim"] + m["rot_dim"]), m["q_rank"]), "sharp"
            else:
                t[p + "q"] = (H * (m["dim"] + m["rot_dim"]), W), "sharp"
            t[p + "dkv"], t[p + "dkv.norm"] = ((r + m["rot_dim"], W), "in"), ((r,), "norm")
            t[p + "uk"], t[p + "uv"] = ((H * m["dim"], r), "in"), ((H * m["vdim"], r), "in")
            t[p + "o"], t[p + "g"] = ((W, H * m["vdim"]), "out"), ((H, W), "in")
        elif kind == "delta":
            D, E, H = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
            t[p + "q"] = t[p + "k"] = (D, W), "in"
            t[p + "v"] = t[p + "g"] = (E, W), "in"
            t[p + "q.conv"] = t[p + "k.conv"] = (D, m["conv"]), 0.5
            t[p + "v.conv"] = (E, m["conv"]), 0.5
            t[p + "b"] = t[p + "a"] = (H, W), "in"
            t[p + "dt_bias"], t[p + "A_log"] = ((H,), "step"), ((H,), "decay")
            t[p + "norm"], t[p + "o"] = ((m["vdim"],), "norm"), ((W, E), "out")
        elif kind == "mingru":
            t[p + "z"] = t[p + "x"] = t[p + "g"] = (m["width"], W), "in"
            t[p + "z.b"] = t[p + "x.b"] = (m["width"],), 0.5
            t[p + "o"] = (W, m["width"]), "in"
        else:
            q, k, v = m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["kv_heads"] * m["vdim"]
            t[p + "q"], t[p + "q.norm"], t[p + "pb"] = ((q, W), "in"), ((q,), "norm"), ((m["heads"],), "few")
            if "kv_from" not in m:
                t[p + "k"], t[p + "v"], t[p + "k.norm"] = ((k, W), "in"), ((v, W), "in"), ((k,), "norm")
            t[p + "o"] = (W, m["heads"] * m["vdim"]), "in"
        if c["architecture"] == "Novosun":
            t[f"l{i}.norm1b"] = t[f"l{i}.norm2b"] = (W,), "norm"
        if c["architecture"] == "Noresun":
            t[f"l{i}.rg1"] = t[f"l{i}.rg2"] = (W, W), "in"
            t[f"l{i}.rg1.b"] = t[f"l{i}.rg2.b"] = (W,), 0.1
        p = f"l{i}.mlp."
        if f["kind"] == "moe":
            E, F = f["router"]["experts"], f["expert"]["ff"]
            t[p + "router"], t[p + "router.b"] = ((E, W), 12.0 / math.sqrt(W)), ((E,), 0.1)
            for e in range(E):
                t[f"{p}e{e}.up"], t[f"{p}e{e}.down"] = ((F, W), "in"), ((W, F), "in")
        else:
            if "limit" in f:
                t[p + "gate"] = (f["ff"], W), "in"
            t[p + "up"], t[p + "down"] = ((f["ff"], W), "in"), ((W, f["ff"]), "out")
    t["final.norm"] = (W,), "norm"
    if c["architecture"] == "Novosun":
        t["head"] = (V, W), "sharp"
    return t


def weights_of(case, seed):
    """The model's tensors on the GPU, drawn from the seed, in the case's data type."""
    c = config_of(case)
    g = torch.Generator(device=GPU).manual_seed(7919 * int(seed) + 1)
    depth = math.sqrt(2.0 * case["layers"])
    kept = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    out = {}
    for name, (shape, how) in tensors_of(c).items():
        if how == "decay":                       # log of a decay rate between 1 and 16
            x = torch.rand(shape, generator=g, device=GPU).mul_(15.0).add_(1.0).log_()
        elif how == "step":                      # what softplus makes a step between 0.001 and 0.1 of
            x = torch.exp(torch.rand(shape, generator=g, device=GPU) * math.log(100.0) + math.log(0.001)).expm1_().log_()
        elif how == "few":                       # sigmoid weights that are not normed over the keys: most of them small
            x = torch.randn(shape, generator=g, device=GPU).sub_(5.0)
        else:
            wide = {"norm": 0.1, "in": shape[-1] ** -0.5, "sharp": 1.2 * shape[-1] ** -0.5, "out": shape[-1] ** -0.5 / depth}
            x = torch.randn(shape, generator=g, device=GPU).mul_(wide.get(how, how) if isinstance(how, str) else how)
            if how == "norm":
                x.add_(1.0)
        out[name] = x.to(kept)
    return out


# -- the passes -------------------------------------------------------------------------------------------------------

def ragged(total, n):
    """n lengths around total / n, from 0.4 to 1.6 times that, in no order."""
    mean = total / n
    even = [max(1, round(mean * (0.4 + 1.2 * (i + 0.5) / n))) for i in range(n)] if n > 1 else [total]
    random.Random(n).shuffle(even)
    return even


def plan_of(case):
    """(lengths of the cached requests, lengths of the new prompts, steps).  A step is a list of (key, first position, count,
    wanted): every decoding request brings one token a step and wants its logits; the new prompts come one after the other,
    `portion` tokens a step in all, and want the logits of their last token."""
    cached = ragged(case["cached"], case["decoding"]) if case["decoding"] else []
    prompts = ragged(case["prompted"], case["prompts"]) if case["prompts"] else []
    steps, cursor = [], [0] * len(prompts)
    while True:
        entries, left = [], case["portion"]
        for i, n in enumerate(prompts):
            take = min(left, n - cursor[i])
            if take:
                entries.append((f"p{i}", cursor[i], take, cursor[i] + take == n))
                cursor[i] += take
                left -= take
        if not entries and len(steps) >= case["steps"]:
            return cached, prompts, steps
        steps.append([(f"d{i}", n + len(steps), 1, True) for i, n in enumerate(cached)] + entries)


def tokens_of(case, seed):
    """{key: all the tokens a request will have by the end of the pass}."""
    cached, prompts, steps = plan_of(case)
    c = config_of(case)
    rng = np.random.default_rng([int(seed), 3])
    vocab = c.get("vocab_size") or c["vocab"]
    return {**{f"d{i}": rng.integers(0, vocab, n + len(steps), dtype=np.int32) for i, n in enumerate(cached)},
            **{f"p{i}": rng.integers(0, vocab, n, dtype=np.int32) for i, n in enumerate(prompts)}}


def listed():
    def case(name, model, layers, dtype="bfloat16", decoding=0, cached=0, steps=0, prompts=0, prompted=0, portion=1, temperature=0.0):
        return dict(name=name, model=model, layers=layers, dtype=dtype, decoding=decoding, cached=cached, steps=steps,
                    prompts=prompts, prompted=prompted, portion=portion, temperature=temperature)
    return [
        # one user chatting with the smallest model: nothing but launches and latency
        case("135m-decode-1", "smollm2-135m", 30, decoding=1, cached=119, steps=16),
        # a small batch of it a few thousand tokens in: the benchmark's default workload
        case("135m-decode-8", "smollm2-135m", 30, decoding=8, cached=8 * 2048, steps=16),
        # one prompt of ordinary length, whole
        case("135m-prompt", "smollm2-135m", 30, prompts=1, prompted=1777, portion=2048),
        # the 32-bit path: two requests sampling at a temperature while a short prompt arrives in portions
        case("135m-float32", "smollm2-135m", 30, "float32", decoding=2, cached=700, steps=6, prompts=1, prompted=333, portion=128, temperature=0.8),
        # a full batch of requests of mixed lengths, nothing arriving
        case("1.7b-decode-64", "smollm2-1.7b", 24, decoding=64, cached=64 * 1216, steps=4),
        # serving: requests decode while prompts arrive in portions
        case("1.7b-serving", "smollm2-1.7b", 24, decoding=37, cached=37 * 900, steps=3, prompts=3, prompted=2611, portion=1024),
        # a long prompt in portions of 2,048 at the layer sizes of the largest model (a quarter of its layers, here and below)
        case("8b-prompt", "llama-3-8b", 8, prompts=1, prompted=5003, portion=2048),
        # long contexts at those sizes
        case("8b-decode-12", "llama-3-8b", 8, decoding=12, cached=12 * 5000, steps=8),
        # the other designs at the width that the benchmark compares them at: prompts of several users in one step ...
        case("novosun-prompt", "novosun-2048", 4, prompts=3, prompted=2345, portion=4096),
        case("ditazen-prompt", "ditazen-2048", 4, prompts=2, prompted=1999, portion=4096),
        # ... and batches that decode
        case("ditazen-decode-8", "ditazen-2048", 4, decoding=8, cached=8 * 1500, steps=16),
        case("noresun-decode-24", "noresun-2048", 4, decoding=24, cached=24 * 1100, steps=8),
    ]


def draw(rng):
    """A case of the same ranges: any of the models (the designs at widths 1,024 and 2,048), decoding, prompts or both."""
    def size(low, high):
        return round(math.exp(rng.uniform(math.log(low), math.log(high))))
    model = rng.choice(["smollm2-135m"] * 2 + ["smollm2-1.7b"] * 2 + ["llama-3-8b"] * 2 +
                       [f"{d}-{w}" for d in ("novosun", "ditazen", "noresun") for w in (1024, 2048)])
    layers = {"smollm2-135m": 30, "smollm2-1.7b": rng.choice([6, 12, 24]), "llama-3-8b": rng.choice([4, 8])}.get(model, 4)
    dtype = "float32" if model == "smollm2-135m" and rng.random() < 0.3 else "bfloat16"
    kind = rng.choice(["decode", "decode", "prompt", "serving"])
    case = dict(model=model, layers=layers, dtype=dtype, decoding=0, cached=0, steps=0, prompts=0, prompted=0, portion=1,
                temperature=rng.choice([0.0, 0.8]) if dtype == "float32" else 0.0)
    most = 512 if dtype == "float32" else 4096
    if kind != "prompt":
        n = size(1, 8 if dtype == "float32" else 64)
        case.update(decoding=n, cached=n * size(32, min(6000, max(64, 77000 // n))), steps=rng.choice([4, 8, 16]) if kind == "decode" else rng.choice([2, 3]))
    if kind != "decode":
        total = size(24, most)
        case.update(prompts=min(total, rng.choice([1, 1, 2, 3, 5])), prompted=total, portion=rng.choice([256, 1024, 2048]))
    largest = max(work(c)["bytes"] for c in listed())
    while work(case)["bytes"] > largest:              # no more than the largest listed one
        case.update(steps=case["steps"] // 2, cached=max(case["decoding"], case["cached"] // 2), prompted=max(case["prompts"], case["prompted"] // 2))
    return case


def prepare(case, seed):
    """The model, its runner with captured programs, and the requests whose tokens are cached already."""
    from runtime.engine import ModelRunner, StepEntry, build_from_config_dict, parse_dtype
    from runtime.sampling import Sampler
    dtype = parse_dtype(case["dtype"])
    _, _, model = build_from_config_dict(config_of(case))
    model.bind(weights_of(case, seed), dtype, torch.device(GPU))
    cached, prompts, steps = plan_of(case)
    tokens = tokens_of(case, seed)
    pages = sum(2 * (-(-(n + len(steps)) // PAGE) + 1) for n in cached) + sum(-(-n // PAGE) for n in prompts) + 8
    runner = ModelRunner(model, n_pages=pages, page_size=PAGE, max_requests=2 * len(cached) + len(prompts), execution="graph")
    room, waiting = 4096 if case["dtype"] == "bfloat16" else 512, []
    for i, n in enumerate(cached):
        runner.create(f"base{i}")
        waiting += [(i, at, min(room, n - at)) for at in range(0, n, room)]
    while waiting:                      # cached in steps of at most `room` tokens, a request at most once a step
        entries, total = [], 0
        for item in list(waiting):
            i, at, n = item
            if total + n <= room and runner.length(f"base{i}") == at:
                entries.append(StepEntry(f"base{i}", tokens[f"d{i}"][at:at + n], []))
                total += n
                waiting.remove(item)
        runner.step(entries)
    wanted = [sum(w for *_, w in step) for step in steps]
    return SimpleNamespace(
        runner=runner, sampler=Sampler(), forks=[(f"base{i}", f"d{i}") for i in range(len(cached))],
        fresh=[f"p{i}" for i in range(len(prompts))],
        steps=[[(key, tokens[key][at:at + n] if n > 1 else [int(tokens[key][at])], [n - 1] if want else []) for key, at, n, want in step]
               for step in steps],
        params=[[(case["temperature"], 11 + r, i) for r in range(n)] for i, n in enumerate(wanted)],
        logits=torch.empty(sum(wanted), model.vocab_size, dtype=torch.float32, device=GPU))


def run(state):
    """The steps of the pass: the logits of every wanted place, and of the token picked there (near-ties of bf16 logits make
    another token as good; in 32 bits the tokens themselves)."""
    from runtime.engine import StepEntry
    runner, at, picked, unread = state.runner, 0, [], None
    for base, key in state.forks:
        runner.fork(base, key)
    for key in state.fresh:
        runner.create(key)
    for step, params in zip(state.steps, state.params):
        logits = runner.step([StepEntry(key, tokens, want) for key, tokens, want in step])
        if not params:
            continue
        state.logits[at:at + len(params)].copy_(logits)
        at += len(params)
        latest = runner.pick(state.sampler, logits, params)
        if unread is not None:
            picked += unread.tokens()
        unread = latest
    picked += unread.tokens()
    for _, key in state.forks:
        runner.release(key)
    for key in state.fresh:
        runner.release(key)
    tokens = torch.tensor(picked, device=GPU)
    out = {"logits": state.logits, "picked": state.logits.gather(1, tokens[:, None])}
    return out if runner.model.dtype == torch.bfloat16 else {**out, "tokens": tokens}


def work(case):
    """Every weight that a step uses, the cached keys and states it reads and the logits, once a step."""
    c, total = config_of(case), {"bytes": 0.0, "flops": 0.0}
    item = 4 if case["dtype"] == "float32" else 2
    shapes = {n: s for n, (s, _) in tensors_of(c).items()}
    llama = "hidden_size" in c
    head = shapes.get("lm_head.weight") or shapes.get("head") or shapes.get("model.embed_tokens.weight") or shapes.get("embed")
    tables = ("model.embed_tokens.weight", "embed", "bigram", "lm_head.weight", "head")
    experts = sum(math.prod(s) for n, s in shapes.items() if ".mlp.e" in n)
    dense = sum(math.prod(s) for n, s in shapes.items() if n not in tables and ".mlp.e" not in n)
    kinds = [dict(type="llama")] * case["layers"] if llama else c["layers"]
    for step in plan_of(case)[2]:
        rows, wanted = sum(n for _, _, n, _ in step), sum(w for *_, w in step)
        total["bytes"] += item * (dense + experts * min(1.0, rows * 2 / 16) + math.prod(head)) + 4 * wanted * head[0]
        total["flops"] += 2.0 * rows * (dense + experts * 2 / 16) + 2.0 * wanted * math.prod(head)
        for layer in kinds:
            m, kind = layer.get("mixer"), layer["type"]
            if kind == "parallel":
                state = m["right"]["heads"] * m["right"]["vdim"] * m["right"]["state"]
                m = m["left"]
            else:
                state = {"gla": lambda: m["heads"] * m["dim"] * m["vdim"], "delta": lambda: m["heads"] * m["dim"] * m["vdim"],
                         "mingru": lambda: m["width"]}.get(kind, lambda: 0)()
            total["bytes"] += 8.0 * state * len(step)
            total["flops"] += 6.0 * state * rows
            if llama:
                heads, score, value = c["num_attention_heads"], c["head_dim"], c["head_dim"]
                a_token, window = 2 * c["num_key_value_heads"] * c["head_dim"], None
            elif kind.startswith("latent"):
                heads, score, value, a_token = m["heads"], m["kv_rank"] + m["rot_dim"], m["kv_rank"], m["kv_rank"] + m["rot_dim"]
                window = (m.get("mask") or {}).get("size")
            elif kind in ("attention", "parallel"):
                heads, score, value, a_token = m["heads"], m["dim"], m["vdim"], m["kv_heads"] * (m["dim"] + m["vdim"])
                window = (m.get("mask") or {}).get("size")
            else:
                continue
            for _, at, n, _ in step:
                total["bytes"] += item * a_token * (min(at, window or at) + n)
                total["flops"] += 2.0 * heads * (score + value) * sum(min(p + 1, window or p + 1) for p in range(at, at + n))
    return total


def tolerance(case):
    """About four times what the logits are off the 64-bit ones: 2.5e-6 in 32 bits, 0.005 to 0.015 in bf16 (less than four
    times that, as a wrong row among many would show as no more)."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-4, "differ": 0.01}
    return {"rel": 0.03, "max": 0.5}


# -- the same in 64 bits ----------------------------------------------------------------------------------------------

def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _centred(x, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps)


def _rotate(x, positions, frequencies, pairs, factor=1.0):
    """The first coordinates of [B, T, heads, n] turn: pair i is (i, i + half), or (2i, 2i + 1) with `pairs`."""
    angle = positions[:, None] * frequencies
    cos, sin = (angle.cos() * factor)[:, None], (angle.sin() * factor)[:, None]
    half, x = len(frequencies), x.clone()
    a, b = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if pairs else (slice(0, half), slice(half, 2 * half))
    u, v = x[..., a].clone(), x[..., b].clone()
    x[..., a], x[..., b] = u * cos - v * sin, v * cos + u * sin
    return x


def _frequencies(base, dims):
    return base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=GPU) / dims)


def _attention(q, k, v, scale, window=None, bias=None):
    """[B, T, H, D] queries over [B, T, G, D] keys, causal; softmax, or with `bias` sigmoid weights that are not normed."""
    B, T, H, _ = q.shape
    each, out = H // k.shape[2], q.new_zeros(B, T, H, v.shape[-1])
    for b in range(B):
        for g in range(k.shape[2]):
            heads = slice(g * each, (g + 1) * each)
            for at in range(0, T, 1024):
                end = min(at + 1024, T)
                low = 0 if window is None else max(0, at - window + 1)
                s = torch.matmul(q[b, at:end, heads].transpose(0, 1).contiguous(), k[b, low:end, g].t().contiguous()) * scale
                i, j = torch.arange(at, end, device=GPU)[:, None], torch.arange(low, end, device=GPU)[None]
                hidden = (j > i) if window is None else (j > i) | (i - j >= window)
                if bias is None:
                    s = s.masked_fill(hidden, float("-inf")).softmax(-1)
                else:
                    s = torch.sigmoid(s + bias[heads, None, None]).masked_fill(hidden, 0.0)
                out[b, at:end, heads] = torch.matmul(s, v[b, low:end, g].contiguous()).transpose(0, 1)
    return out


def _conv(x, taps):
    n = taps.shape[1]
    padded = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    return sum(padded[:, j:j + x.shape[1]] * taps[:, j] for j in range(n))


def _scan(q, k, v, decay, beta=None):
    """S <- decay S; u = v, or with `beta` beta (v - S^T k); S <- S + k u^T; o = S^T q, row by row, for [B, T, H, ...]; a
    decay a row ([B, T, H, 1]) or a channel of the key."""
    B, T, H, D = k.shape
    S, out = q.new_zeros(B, H, D, v.shape[-1]), torch.empty_like(v)
    for t in range(T):
        S = S * decay[:, t, :, :, None]
        u = v[:, t] if beta is None else beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
        S.addcmul_(k[:, t, :, :, None], u[:, :, None])
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    return out


class _Exact:
    def __init__(self, case, seed):
        self.c, self.w = config_of(case), weights_of(case, seed)

    def t(self, name):
        return self.w[name].double()

    def linear(self, x, name, bias=None):
        y = x @ self.t(name).t()
        return y if bias is None else y + self.t(bias)

    def norm(self, x, name, eps):
        return _rms(x, eps) * self.t(name)

    def llama(self, ids):
        c, B, T = self.c, *ids.shape
        H, G, D, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"]
        x, pos, f = self.w["model.embed_tokens.weight"][ids].double(), torch.arange(T, device=GPU, dtype=torch.float64), _frequencies(c["rope_theta"], D)
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.norm(x, p + "input_layernorm.weight", eps)
            q = _rotate(self.linear(h, p + "self_attn.q_proj.weight").view(B, T, H, D), pos, f, False)
            k = _rotate(self.linear(h, p + "self_attn.k_proj.weight").view(B, T, G, D), pos, f, False)
            v = self.linear(h, p + "self_attn.v_proj.weight").view(B, T, G, D)
            x = x + self.linear(_attention(q, k, v, D ** -0.5).flatten(2), p + "self_attn.o_proj.weight")
            h = self.norm(x, p + "post_attention_layernorm.weight", eps)
            h = torch.nn.functional.silu(self.linear(h, p + "mlp.gate_proj.weight")) * self.linear(h, p + "mlp.up_proj.weight")
            x = x + self.linear(h, p + "mlp.down_proj.weight")
        return self.norm(x, "model.norm.weight", eps), "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"

    def novosun(self, ids):
        c, eps = self.c, self.c["norm"]["eps"]
        x = self.w["embed"][ids].double()
        for i, layer in enumerate(c["layers"]):
            mix = self.novosun_side if layer["type"] == "parallel" else self.novosun_gla
            y = mix(self.norm(x, f"l{i}.norm1", eps), f"l{i}.mix.", layer["mixer"], eps)
            x = x + c["residual_mult"] * self.norm(y, f"l{i}.norm1b", eps)
            h, limit, p = self.norm(x, f"l{i}.norm2", eps), layer["mlp"]["limit"], f"l{i}.mlp."
            g, u = self.linear(h, p + "gate").clamp(max=limit), self.linear(h, p + "up").clamp(-limit, limit)
            x = x + c["residual_mult"] * self.norm(self.linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down"), f"l{i}.norm2b", eps)
        return self.norm(x, "final.norm", eps), "head"

    def novosun_gla(self, h, p, m, eps):
        B, T, H = *h.shape[:2], m["heads"]
        q, k = (self.linear(h, p + n).view(B, T, H, m["dim"]) for n in "qk")
        z = self.linear(self.linear(h, p + "a1"), p + "a2", p + "a2.b").view(B, T, H, m["dim"])
        o = _scan(q * m["dim"] ** -0.5, k, self.linear(h, p + "v").view(B, T, H, m["vdim"]), torch.sigmoid(z) ** (1.0 / m["tau"]))
        return self.linear(self.norm(o, p + "norm", eps).flatten(2) * torch.nn.functional.silu(self.linear(h, p + "g")), p + "o")

    def novosun_side(self, h, p, m, eps):
        B, T = h.shape[:2]
        a, s = m["left"], m["right"]
        q = self.norm(self.linear(h, p + "left.q").view(B, T, a["heads"], a["dim"]), p + "left.q.norm", eps)
        k = self.norm(self.linear(h, p + "left.k").view(B, T, a["kv_heads"], a["dim"]), p + "left.k.norm", eps)
        o = _attention(q, k, self.linear(h, p + "left.v").view(B, T, a["kv_heads"], a["vdim"]), a["scale"])
        left = self.linear((o * torch.sigmoid(self.linear(h, p + "left.g"))[..., None]).flatten(2), p + "left.o")
        H, V, N, G = s["heads"], s["vdim"], s["state"], s["groups"]
        z, xbc, dt = self.linear(h, p + "right.in").split([H * V, H * V + 2 * G * N, H], -1)
        xbc = torch.nn.functional.silu(_conv(xbc, self.t(p + "right.conv")) + self.t(p + "right.conv.b"))
        x, b, r = xbc.split([H * V, G * N, G * N], -1)
        x, b, r = x.reshape(B, T, H, V), *(y.reshape(B, T, G, N).repeat_interleave(H // G, 2) for y in (b, r))
        dt = torch.nn.functional.softplus(dt + self.t(p + "right.dt_bias"))[..., None]
        y = _scan(r, b, dt * x, torch.exp(-self.t(p + "right.A_log").exp()[:, None] * dt)) + self.t(p + "right.D")[:, None] * x
        y = y.reshape(B, T, H * V) * torch.nn.functional.silu(z)
        y = _rms(y.reshape(B, T, s["norm_groups"], -1), eps).reshape(B, T, H * V) * self.t(p + "right.norm")
        return 0.5 * (self.norm(left, p + "left.out", eps) + self.norm(self.linear(y, p + "right.o"), p + "right.out", eps))

    def ditazen(self, ids):
        c, eps = self.c, self.c["norm"]["eps"]
        x = self.w["embed"][ids].double()
        for i, layer in enumerate(c["layers"]):
            mix = self.ditazen_delta if layer["type"] == "delta" else self.ditazen_latent
            x = x + mix(_centred(x, eps) * self.t(f"l{i}.norm1"), f"l{i}.mix.", layer["mixer"], eps)
            h = torch.nn.functional.gelu(self.linear(_centred(x, eps) * self.t(f"l{i}.norm2"), f"l{i}.mlp.up"))
            x = x + self.linear(h, f"l{i}.mlp.down")
        return _centred(x, eps) * self.t("final.norm") * c["logit_scale"], "embed"

    def ditazen_latent(self, h, p, m, eps):
        B, T, H, D, r, rot = *h.shape[:2], m["heads"], m["dim"], m["kv_rank"], m["rot"]
        second, dims = "q_rank" in m, rot["dims"]
        f, factor, s = _frequencies(rot["base"], dims), 1.0, rot.get("scaling")
        if s:
            at = lambda turns: dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))  # noqa: E731
            low, high = max(math.floor(at(s["fast"])), 0), min(math.ceil(at(s["slow"])), dims - 1)
            ramp = ((torch.arange(dims // 2, device=GPU, dtype=torch.float64) - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
            f, factor = f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0
        q = self.linear(self.norm(self.linear(h, p + "dq"), p + "dq.norm", eps), p + "uq") if second else self.linear(h, p + "q")
        q = q.view(B, T, H, D + m["rot_dim"])
        pos = torch.arange(T, device=GPU, dtype=torch.float64)
        q = torch.cat((q[..., :D], _rotate(q[..., D:], pos, f, second, factor)), -1)
        dkv = self.linear(h, p + "dkv")
        latent = self.norm(dkv[..., :r], p + "dkv.norm", eps)
        turned = _rotate(dkv[:, :, None, r:], pos, f, second, factor).expand(B, T, H, m["rot_dim"])
        k = torch.cat((self.linear(latent, p + "uk").view(B, T, H, D), turned), -1)
        o = _attention(q, k, self.linear(latent, p + "uv").view(B, T, H, m["vdim"]), m["scale"], (m.get("mask") or {}).get("size"))
        return self.linear((o * torch.sigmoid(self.linear(h, p + "g"))[..., None]).flatten(2), p + "o")

    def ditazen_delta(self, h, p, m, eps):
        B, T, H, G = *h.shape[:2], m["heads"], m["kv_heads"]
        q, k, v = (torch.nn.functional.silu(_conv(self.linear(h, p + n), self.t(p + n + ".conv"))) for n in "qkv")
        q, k = (y.view(B, T, G, m["dim"]) for y in (q, k))
        q, k = (y * torch.rsqrt(y.square().sum(-1, keepdim=True) + 1e-6) for y in (q, k))
        q, k = (y.repeat_interleave(H // G, 2) for y in (q * m["dim"] ** -0.5, k))
        decay = torch.exp(-self.t(p + "A_log").exp() * torch.nn.functional.softplus(self.linear(h, p + "a", p + "dt_bias")))
        o = _scan(q, k, v.view(B, T, H, m["vdim"]), decay[..., None], torch.sigmoid(self.linear(h, p + "b")))
        return self.linear(self.norm(o, p + "norm", eps).flatten(2) * torch.nn.functional.silu(self.linear(h, p + "g")), p + "o")

    def noresun(self, ids):
        c, eps, alpha = self.c, self.c["norm"]["eps"], self.c["postln_alpha"]
        e = c["embedding"]["bigram"]
        before = torch.cat((torch.zeros_like(ids[:, :1]), ids[:, :-1]), 1)
        pair = (before * e["mul_prev"] + ids * e["mul_cur"]) % e["buckets"]
        pair[:, 0] = e["buckets"]
        x = self.w["embed"][ids].double() * c["embedding"]["scale"] + self.w["bigram"][pair].double()
        kept = {}
        for i, layer in enumerate(c["layers"]):
            p = f"l{i}."
            y = self.noresun_unit(x, p + "mix.") if layer["type"] == "mingru" else self.noresun_attention(x, i, layer["mixer"], eps, kept)
            x = self.norm(alpha * x + y * torch.sigmoid(self.linear(x, p + "rg1", p + "rg1.b")), p + "norm1", eps)
            y = self.noresun_experts(x, p + "mlp.", layer["mlp"]["router"])
            x = self.norm(alpha * x + y * torch.sigmoid(self.linear(x, p + "rg2", p + "rg2.b")), p + "norm2", eps)
        return self.norm(x, "final.norm", eps), "embed"

    def noresun_unit(self, h, p):
        z = torch.sigmoid(self.linear(h, p + "z", p + "z.b"))
        u = self.linear(h, p + "x", p + "x.b")
        u = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
        S, out = torch.zeros_like(u[:, 0]), torch.empty_like(u)
        for t in range(h.shape[1]):
            S = torch.lerp(S, u[:, t], z[:, t])
            out[:, t] = S
        return self.linear(out * torch.nn.functional.silu(self.linear(h, p + "g")), p + "o")

    def noresun_attention(self, h, i, m, eps, kept):
        B, T, p, rot, s = *h.shape[:2], f"l{i}.mix.", m["rot"], m["rot"]["scaling"]
        f = _frequencies(rot["base"], rot["dims"])
        wave = 2.0 * math.pi / f                  # the long wavelengths are slowed down, with a ramp between
        ramp = ((s["original"] / wave - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
        f, pos = (1.0 - ramp) * f / s["factor"] + ramp * f, torch.arange(T, device=GPU, dtype=torch.float64)
        if "kv_from" not in m:
            k = self.norm(self.linear(h, p + "k"), p + "k.norm", eps).view(B, T, m["kv_heads"], m["dim"])
            kept[i] = _rotate(k, pos, f, True), self.linear(h, p + "v").view(B, T, m["kv_heads"], m["vdim"])
        q = _rotate(self.norm(self.linear(h, p + "q"), p + "q.norm", eps).view(B, T, m["heads"], m["dim"]), pos, f, True)
        k, v = kept[m.get("kv_from", i)]
        return self.linear(_attention(q, k, v, m["scale"], m["mask"]["size"], self.t(p + "pb")).flatten(2), p + "o")

    def noresun_experts(self, x, p, router):
        logits = self.linear(x, p + "router", p + "router.b")
        best, which = logits.topk(router["top"], -1)
        gate, out = best.softmax(-1), torch.zeros_like(x)
        for e in range(router["experts"]):
            rows = (which == e).any(-1)
            share = torch.where(which == e, gate, 0.0).sum(-1)[rows][:, None]
            out[rows] += share * self.linear(self.linear(x[rows], f"{p}e{e}.up").relu().square(), f"{p}e{e}.down")
        return out


def exact(case, seed):
    """The logits in 64 bits: every request's whole sequence at once, a few requests at a time, padded at the end."""
    model = _Exact(case, seed)
    forward = getattr(model, "llama" if case["model"] in LLAMA else case["model"].split("-")[0])
    tokens = tokens_of(case, seed)
    places = [(key, at + n - 1) for step in plan_of(case)[2] for key, at, n, want in step if want]
    logits, keys = {}, sorted(tokens, key=lambda k: len(tokens[k]))
    while keys:
        longest = len(tokens[keys[-1]])
        some = keys[-max(1, 16384 // longest):]
        keys = keys[:-len(some)]
        ids = torch.zeros(len(some), longest, dtype=torch.int64)
        for b, key in enumerate(some):
            ids[b, :len(tokens[key])] = torch.from_numpy(tokens[key].astype(np.int64))
        hidden, head = forward(ids.to(GPU))
        for b, key in enumerate(some):
            mine = [at for k, at in places if k == key]
            if mine:
                rows = hidden[b, mine] @ model.t(head).t()
                logits.update({(key, at): row for at, row in zip(mine, rows)})
    logits = torch.stack([logits[place] for place in places])
    out = {"logits": logits, "picked": None if case["temperature"] else logits.amax(1, keepdim=True)}
    return out if case["dtype"] == "bfloat16" else {**out, "tokens": None}
