"""The work that is timed when the engine's speed is compared between two versions.

A case is one call sequence that a program on this framework makes, with its sizes: prompts run whole in one step, a
decode step of a batch, a serving step that holds decoded tokens beside a portion of a prompt, and the sampling of a
batch.  Models are random-weights ones at the sizes that the benchmark and the tests use.

`listed()` names the cases, `draw(rng)` gives another one of the same ranges, `prepare` makes what a program holds
before the call, `run` is one pass, `work` what a pass cannot do without, `tolerance` how far two correct
implementations are apart, and `exact` the same outputs in 64 bits from plain torch.
"""
from __future__ import annotations

import math
import zlib

import torch

import easy_gpt  # noqa: F401  (makes easy_gpt.cpp_amd importable)
from easy_gpt.cpp_amd.config.registry import resolve_architecture
from easy_gpt.cpp_amd.engine import Engine, StepEntry
from easy_gpt.cpp_amd.parts.model import build_model
from easy_gpt.cpp_amd.sampling import Sampler, SamplingParams

F64 = torch.float64


# ------------------------------------------------------------------------------------------------------------- models
def _qwen2(layers, hidden, heads, kv_heads, inner, vocab, tied=True, theta=1e6, eps=1e-6, longest=32768):
    return {
        "architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "num_hidden_layers": layers, "hidden_size": hidden,
        "num_attention_heads": heads, "num_key_value_heads": kv_heads, "intermediate_size": inner, "vocab_size": vocab,
        "rope_theta": theta, "rms_norm_eps": eps, "tie_word_embeddings": tied, "max_position_embeddings": longest,
        "use_sliding_window": False, "hidden_act": "silu", "torch_dtype": "bfloat16",
    }


def _nebanex(width, heads, kv_heads, hd, s_heads, s_dim, s_vdim, experts, top, ff, shared, layers=4, vocab=32768):
    layer = {
        "type": "parallel",
        "mixer": {"left": {"heads": heads, "kv_heads": kv_heads, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "bias_max": 512,
                           "q_temp": {"coef": 0.1, "every": 1024}},
                  "right": {"heads": s_heads, "dim": s_dim, "vdim": s_vdim, "tau": 8.0}},
        "mlp": {"kind": "moe", "router": {"experts": experts, "top": top}, "expert": {"ff": ff}, "shared": {"ff": shared}},
    }
    return {"architecture": "Nebanex", "vocab": vocab, "width": width, "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0},
            "logit_softcap": 50.0, "layers": [layer] * layers}


MODELS = {
    "tiny_a": _qwen2(2, 64, 4, 2, 176, 512, theta=1e4, longest=128),                 # the two tiny test configurations
    "tiny_b": _qwen2(3, 96, 3, 1, 256, 1000, tied=False, eps=1e-5, longest=256),
    "0.5b": _qwen2(24, 896, 14, 2, 4864, 151936),                                    # the sizes of the benchmark
    "1.5b": _qwen2(28, 1536, 12, 2, 8960, 151936),
    "3b": _qwen2(36, 2048, 16, 2, 11008, 151936),
    "7b": _qwen2(28, 3584, 28, 4, 18944, 152064, tied=False),
    "nebanex_w896": _nebanex(896, 14, 2, 64, 7, 64, 128, 16, 4, 1024, 768),          # and of its other design with experts
    "nebanex_w2048": _nebanex(2048, 16, 4, 128, 16, 64, 128, 32, 4, 1536, 2048),
}
BIAS_ROWS, DECAY_RANK = 32, 16       # the Nebanex tensors' sizes that its configuration does not name


def _is_nebanex(case):
    return case["model"].startswith("nebanex")


def _vocab(case):
    cfg = MODELS[case["model"]]
    return cfg["vocab"] if _is_nebanex(case) else cfg["vocab_size"]


def _position_limit(case):
    return 1 << 20 if _is_nebanex(case) else MODELS[case["model"]]["max_position_embeddings"]


# -------------------------------------------------------------------------------------------------------------- cases
def _prompts(name, model, dtype, requests, shortest, longest):
    return {"name": name, "kind": "prompts", "model": model, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest}


def _decode(name, model, dtype, requests, shortest, longest):
    return {"name": name, "kind": "decode", "model": model, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest}


def _serve(name, model, dtype, requests, shortest, longest, portion):
    return {"name": name, "kind": "serve", "model": model, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest, "portion": portion}


def listed():
    return [
        # the smallest call: three short prompts of the tiny test model in one step, all launches and host time
        _prompts("tiny_prompts", "tiny_a", "float32", 3, 5, 33),
        # interactive decoding, one user, behind a prompt of 2,048 tokens
        _decode("decode_1", "0.5b", "bfloat16", 1, 2048, 2048),
        # the benchmark's decode: eight users, here with conversations of different lengths
        _decode("decode_8", "0.5b", "bfloat16", 8, 1021, 2048),
        # a loaded server: 64 users from short to long conversations
        _decode("decode_64", "0.5b", "bfloat16", 64, 130, 2048),
        # a prompt of the benchmark's length: time to the first token
        _prompts("prompt_2048", "0.5b", "bfloat16", 1, 2048, 2048),
        # a long document in one step, at a length that no tile divides
        _prompts("long_prompt", "0.5b", "bfloat16", 1, 8191, 8191),
        # a step of the mixed serving workload: 40 decoded tokens beside a portion of 512 tokens of a new prompt
        _serve("serve_1.5b", "1.5b", "bfloat16", 40, 128, 2048, 512),
        # a model whose weights are the step: 7B sizes, eight users
        _decode("decode_7b", "7b", "bfloat16", 8, 500, 1400),
        # and a prompt there: dense matrix products
        _prompts("prompt_7b", "7b", "bfloat16", 1, 2048, 2048),
        # the true 32-bit path: three prompts of odd lengths together
        _prompts("prompts_f32", "0.5b", "float32", 3, 301, 907),
        # the design with experts, a distance bias and a decaying matrix state: three prompts together
        _prompts("nebanex_prompts", "nebanex_w896", "bfloat16", 3, 333, 1357),
        # sampling with the default options over the whole vocabulary for 64 users
        {"name": "sample_64", "kind": "sample", "requests": 64, "vocab": 151936, "temperature": 0.8, "top_k": 20, "top_p": 0.95},
    ]


def _log(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49))))))


# Resident tokens of a drawn decode or serving case, and tokens of its prompts, are bounded per model.
_RESIDENT = {"tiny_a": 600, "tiny_b": 1500, "0.5b": 80000, "1.5b": 24000, "3b": 12000, "7b": 9000, "nebanex_w896": 24000, "nebanex_w2048": 12000}
_TOKENS = {"tiny_a": 300, "tiny_b": 800, "0.5b": 9000, "1.5b": 6000, "3b": 3500, "7b": 2040, "nebanex_w896": 5000, "nebanex_w2048": 3000}


def draw(rng):
    """Kinds by how often a program meets them; sizes over the whole range."""
    kind = rng.choices(["decode", "prompts", "serve", "sample"], [4, 4, 2, 1])[0]
    if kind == "sample":
        return {"kind": "sample", "requests": _log(rng, 1, 64), "vocab": rng.choice([32768, 151936, 152064]),
                "temperature": rng.choice([0.0, 0.6, 0.8, 1.0]), "top_k": rng.choice([0, 20, 50]), "top_p": rng.choice([0.8, 0.95, 1.0])}
    models = ["0.5b", "1.5b", "3b", "7b", "tiny_a", "tiny_b", "nebanex_w896", "nebanex_w2048"]
    model = rng.choices(models, [6, 3, 2, 2, 1, 1, 2, 1])[0]
    if model.startswith("tiny"):
        dtype = "float32"
    else:
        dtype = "float32" if model == "0.5b" and rng.random() < 0.34 else "bfloat16"
    if kind == "prompts":
        requests, most = _log(rng, 1, 8), _TOKENS[model]
    else:
        requests, most = _log(rng, 1, 64), _RESIDENT[model]
    limit = 100 if model == "tiny_a" else 200 if model == "tiny_b" else 8191 if kind == "prompts" else 4095
    longest = _log(rng, min(17, limit), max(18, min(limit, most // requests)))
    shortest = max(1, int(longest * rng.uniform(0.1, 1.0)))
    if kind == "prompts":
        return {"kind": kind, "model": model, "dtype": dtype, "requests": requests, "shortest": shortest, "longest": longest}
    if model == "tiny_a":
        longest, shortest = min(longest, 64), min(shortest, 64)
    case = {"kind": kind, "model": model, "dtype": dtype, "requests": requests, "shortest": shortest, "longest": longest}
    if kind == "serve":
        case["portion"] = _log(rng, 16, 100 if model.startswith("tiny") else 1024)
    return case


def _lengths(case):
    """The requests' lengths, spread evenly from the shortest to the longest."""
    n, a, b = case["requests"], case["shortest"], case["longest"]
    return [b] if n == 1 else [a + (b - a) * i // (n - 1) for i in range(n)]


def _room(case):
    """Tokens that a decoding request of this case may grow by before it ends and its prompt is run again."""
    return min(1024, _position_limit(case) - case["longest"] - 2)


# ------------------------------------------------------------------------------------------------------------- inputs
_NORMS = {"input_layernorm", "post_attention_layernorm", "norm", "norm1", "norm2", "out"}


def _weight(case, seed, name, shape, device="cuda"):
    """The stored tensor `name`: a matrix N(0, 0.36 / inputs), which is N(0, 0.02) at a width of 896 and keeps activations
    of the same size at every width; a table of biases by distance N(0, 0.5); norm weights around one; biases N(0, 0.02)."""
    g = torch.Generator(device=device).manual_seed((int(seed) << 32) + zlib.crc32(name.encode()))
    last = name.removesuffix(".weight").split(".")[-1]
    std = 0.5 if last == "rel" else 0.6 * shape[1] ** -0.5 if len(shape) == 2 else 0.02
    w = torch.randn(tuple(shape), generator=g, device=device, dtype=torch.float32) * std
    if last in _NORMS:
        w += 1.0
    return w.to(torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32)


def _tokens(case, seed, counts):
    """A list of token ids per request: uniform over the vocabulary."""
    g = torch.Generator().manual_seed(int(seed) * 2 + 1)
    return [torch.randint(0, _vocab(case), (n,), generator=g).tolist() for n in counts]


def _all_tokens(case, seed):
    """Every request's tokens: its prompt, and for requests that decode those that it is fed afterwards; at the end the
    serving step's portion."""
    grow = 0 if case["kind"] == "prompts" else _room(case) + 1
    counts = [n + grow for n in _lengths(case)]
    return _tokens(case, seed, counts + ([case["portion"]] if case["kind"] == "serve" else []))


def _logits(case, seed, device="cuda"):
    """Logits as a model gives them: wide, with a few likely tokens in every row."""
    g = torch.Generator(device=device).manual_seed(int(seed))
    r, v = case["requests"], case["vocab"]
    x = torch.randn((r, v), generator=g, device=device, dtype=torch.float32) * 2.5
    likely = torch.randint(0, v, (r, 12), generator=g, device=device)
    return x.scatter_add_(1, likely, torch.rand((r, 12), generator=g, device=device) * 12)


def _model(case, seed):
    config = MODELS[case["model"]]
    arch = resolve_architecture(config)
    typed = arch.config_class.from_dict(config, where="config")
    model = build_model(arch.build_spec(typed))
    shapes = {s.name: s.shape for s in model.param_specs()}
    model.load(lambda name: _weight(case, seed, name, shapes[name]), getattr(torch, case["dtype"]), torch.device("cuda:0"))
    model.config = typed
    return model


FILL = 16384          # tokens of prompts that `_fill` runs in one step


def _fill(state):
    """Puts the decoding requests' prompts into the cache."""
    engine, entries, total = state["engine"], [], 0
    for rid, ids, n in zip(state["ids"], state["tokens"], state["lengths"]):
        engine.add_request(rid)
        entries.append(StepEntry(rid, ids[:n]))
        total += n
        if total + state["lengths"][-1] > FILL or rid == state["ids"][-1]:
            engine.step(entries)
            entries, total = [], 0
    state["grown"] = 0


def prepare(case, seed):
    """The model with its engine, the requests' tokens and, for cases that decode, the prompts in the cache.  One pass
    has been made, as in a program that serves: the step's captured graph exists."""
    if case["kind"] == "sample":
        n = case["requests"]
        t, k, p = case["temperature"], case["top_k"], case["top_p"]
        params = [SamplingParams(greedy=True) if t == 0 else SamplingParams(temperature=t, top_k=k, top_p=p, seed=int(seed) % 1000003)] * n
        return {"kind": "sample", "sampler": Sampler("cuda:0"), "logits": _logits(case, seed), "params": params,
                "serials": list(range(n)), "counts": [(7 * i) % 50 for i in range(n)]}
    lengths, tokens = _lengths(case), _all_tokens(case, seed)
    extra = case.get("portion", 0)
    room = 0 if case["kind"] == "prompts" else _room(case)
    engine = Engine(_model(case, seed), page_size=16, max_tokens=sum(n + room + 32 for n in lengths) + extra + 32,
                    max_requests=case["requests"] + 1)
    state = {"kind": case["kind"], "engine": engine, "lengths": lengths, "tokens": tokens, "room": room,
             "ids": ["r%d" % i for i in range(len(lengths))]}
    if case["kind"] == "prompts":
        state["entries"] = [StepEntry(rid, ids, [len(ids) - 1]) for rid, ids in zip(state["ids"], tokens)]
    else:
        _fill(state)
    run(state)
    return state


def run(state):
    """One pass.  Prompts: admit the requests, run them in one step, let them go; logits behind the last tokens.
    Decode: one token per request (given ones, so that two implementations stay on the same texts); logits of every
    row.  Serve: the same beside the first portion of a new request.  Sample: tokens on the device."""
    if state["kind"] == "sample":
        return state["sampler"].sample_async(state["logits"], state["params"], state["serials"], state["counts"]).device
    engine = state["engine"]
    if state["kind"] == "prompts":
        for rid in state["ids"]:
            engine.add_request(rid)
        logits = engine.step(state["entries"])
        for rid in state["ids"]:
            engine.finish(rid)
        return logits
    if state["grown"] >= state["room"]:                    # the conversations end and begin again
        for rid in state["ids"]:
            engine.finish(rid)
        _fill(state)
    at = state["grown"]
    entries = [StepEntry(rid, (ids[n + at],), (0,)) for rid, ids, n in zip(state["ids"], state["tokens"], state["lengths"])]
    if state["kind"] == "serve":
        engine.add_request("new")
        entries.append(StepEntry("new", state["tokens"][-1], (len(state["tokens"][-1]) - 1,)))
    logits = engine.step(entries)
    if state["kind"] == "serve":
        engine.finish("new")
    state["grown"] = at + 1
    return logits


# --------------------------------------------------------------------------------------------------------------- work
def _sizes(case):
    """(parameters of the layers that a token uses, all of them but for experts, experts' share, width, vocabulary)."""
    c = MODELS[case["model"]]
    if not _is_nebanex(case):
        h, i, hd = c["hidden_size"], c["intermediate_size"], c["hidden_size"] // c["num_attention_heads"]
        layer = h * hd * (2 * c["num_attention_heads"] + 2 * c["num_key_value_heads"]) + 3 * h * i
        return dict(layers=c["num_hidden_layers"], layer=layer, expert=0, experts=0, top=0, width=h, heads=c["num_attention_heads"],
                    kv=c["num_key_value_heads"], hd=hd, vocab=c["vocab_size"], state=0)
    m, r = c["layers"][0]["mixer"]["left"], c["layers"][0]["mixer"]["right"]
    f, w = c["layers"][0]["mlp"], c["width"]
    left = w * m["dim"] * (3 * m["heads"] + 2 * m["kv_heads"])
    right = w * r["heads"] * (2 * r["dim"] + 3 * r["vdim"]) + DECAY_RANK * (w + r["heads"] * r["dim"])
    layer = left + right + 3 * w * f["shared"]["ff"] + w * f["router"]["experts"]
    return dict(layers=len(c["layers"]), layer=layer, expert=3 * w * f["expert"]["ff"], experts=f["router"]["experts"],
                top=f["router"]["top"], width=w, heads=m["heads"], kv=m["kv_heads"], hd=m["dim"], vocab=c["vocab"],
                state=r["heads"] * r["dim"] * r["vdim"])


def work(case):
    if case["kind"] == "sample":
        n = case["requests"] * case["vocab"]
        return {"bytes": 4 * n + 4 * case["requests"], "flops": 2 * n}
    s, size = _sizes(case), 2 if case["dtype"] == "bfloat16" else 4
    lengths = _lengths(case)
    if case["kind"] == "prompts":
        tokens, rows, requests = sum(lengths), len(lengths), len(lengths)
        pairs, held = sum(n * (n + 1) // 2 for n in lengths), 0
    else:
        lengths = [n + 2 for n in lengths]
        tokens = rows = requests = len(lengths)
        pairs, held = sum(lengths), sum(lengths) - len(lengths)
        if case["kind"] == "serve":
            p = case["portion"]
            tokens, rows, requests, pairs = tokens + p, rows + 1, requests + 1, pairs + p * (p + 1) // 2
    read = min(s["experts"], tokens * s["top"])
    weights = s["layers"] * (s["layer"] + read * s["expert"]) + s["vocab"] * s["width"]
    kv = 2 * s["layers"] * s["kv"] * s["hd"] * (held + tokens)
    state = 4 * s["layers"] * s["state"] * requests * (1 if case["kind"] == "prompts" else 2)
    per_token = 2 * s["layers"] * (s["layer"] + s["top"] * s["expert"] + 3 * s["state"])
    return {"bytes": size * (weights + kv + tokens * s["width"]) + state + 4 * rows * s["vocab"],
            "flops": tokens * per_token + 2 * rows * s["vocab"] * s["width"] + 4 * s["layers"] * s["heads"] * s["hd"] * pairs}


def tolerance(case):
    """About four times the largest error against `exact` that was seen: 7.6e-7 in float32; in bfloat16 5.4e-3 for the Qwen2
    sizes, and 8e-3 to 2e-2 with experts, where rounding may turn the choice between two nearly equal ones."""
    if case["kind"] == "sample":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 3e-2, "max": 5e-1} if _is_nebanex(case) else {"rel": 2e-2, "max": 3e-1}


# -------------------------------------------------------------------------------------------------------- in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def _causal(q, k, v, scale, bias=None):
    """q [n, heads, d] of the last n tokens, k, v [t, kv heads, d] of all t: causal attention, [n, heads * d].
    bias: [heads, t], added by distance."""
    n, heads, d = q.shape
    t, kv = k.shape[0], k.shape[1]
    keys = k.permute(1, 2, 0).contiguous().repeat_interleave(heads // kv, 0)
    values = v.transpose(0, 1).contiguous().repeat_interleave(heads // kv, 0)
    out = torch.empty((n, heads, v.shape[2]), dtype=q.dtype, device=q.device)
    for a in range(0, n, 512):
        b = min(n, a + 512)
        s = torch.matmul(q[a:b].transpose(0, 1).contiguous(), keys) * scale
        far = torch.arange(t - n + a, t - n + b, device=q.device)[:, None] - torch.arange(t, device=q.device)[None]
        if bias is not None:
            s += bias[:, far.clamp(min=0)]
        s.masked_fill_(far < 0, -math.inf)
        out[a:b] = torch.matmul(torch.softmax(s, -1), values).transpose(0, 1)
    return out.reshape(n, -1)


def _exact_qwen2(case, seed, texts):
    """Logits behind the last token of every text.  Rotation angles are float32 products, as the model defines them."""
    c = MODELS[case["model"]]
    h, inner, heads, kv, vocab = (c[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads", "num_key_value_heads", "vocab_size"))
    hd, eps = h // heads, c["rms_norm_eps"]
    w = lambda name, *shape: _weight(case, seed, name, shape).to(F64)  # noqa: E731
    embed = _weight(case, seed, "model.embed_tokens.weight", (vocab, h))
    ids = torch.tensor([t for text in texts for t in text], device="cuda")
    starts = [0]
    for text in texts:
        starts.append(starts[-1] + len(text))
    x = embed[ids].to(F64)
    freq = 1.0 / torch.pow(torch.tensor(c["rope_theta"], dtype=torch.float32), 2.0 * torch.arange(hd // 2, dtype=torch.float32) / hd)
    where = torch.cat([torch.arange(len(text)) for text in texts]).to(torch.float32)
    angles = (where[:, None] * freq[None]).to(F64).cuda()
    cos, sin = torch.cos(angles)[:, None], torch.sin(angles)[:, None]

    def rotate(y):
        a, b = y[..., : hd // 2], y[..., hd // 2 :]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    for i in range(c["num_hidden_layers"]):
        p = "model.layers.%d." % i
        y = _rms(x, w(p + "input_layernorm.weight", h), eps)
        q, k, v = (torch.addmm(w(p + "self_attn.%s_proj.bias" % n, m * hd), y, w(p + "self_attn.%s_proj.weight" % n, m * hd, h).t()).view(-1, m, hd)
                   for n, m in (("q", heads), ("k", kv), ("v", kv)))
        q, k = rotate(q), rotate(k)
        o = torch.cat([_causal(q[a:b], k[a:b], v[a:b], hd ** -0.5) for a, b in zip(starts, starts[1:])])
        x += o @ w(p + "self_attn.o_proj.weight", h, heads * hd).t()
        y = _rms(x, w(p + "post_attention_layernorm.weight", h), eps)
        gate, up, down = (w(p + "mlp.%s_proj.weight" % n, *shape).t() for n, shape in (("gate", (inner, h)), ("up", (inner, h)), ("down", (h, inner))))
        for a in range(0, x.shape[0], 16384):
            g = y[a : a + 16384] @ gate
            x[a : a + 16384] += (g * torch.sigmoid(g) * (y[a : a + 16384] @ up)) @ down
    last = torch.tensor([b - 1 for b in starts[1:]], device="cuda")
    y = _rms(x[last], w("model.norm.weight", h), eps)
    head = embed if c["tie_word_embeddings"] else _weight(case, seed, "lm_head.weight", (vocab, h))
    return y @ head.to(F64).t()


def _distance_rows(t, rows, far):
    """The row of the bias table for every distance below t."""
    half = rows // 2
    return torch.tensor([n if n < half else min(rows - 1, half + int(math.floor(math.log(n / half) / math.log(far / half) * (rows - half))))
                         for n in range(t)], device="cuda")


def _exact_nebanex(case, seed, texts):
    c = MODELS[case["model"]]
    width, eps = c["width"], c["norm"]["eps"]
    w = lambda name, *shape: _weight(case, seed, name, shape).to(F64)  # noqa: E731
    embed = _weight(case, seed, "embed", (c["vocab"], width))
    ids = torch.tensor([t for text in texts for t in text], device="cuda")
    lens = [len(text) for text in texts]
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    x = embed[ids].to(F64) * c["embedding"]["scale"]
    where = torch.cat([torch.arange(n) for n in lens]).to("cuda", F64)
    silu = lambda g: g * torch.sigmoid(g)  # noqa: E731
    for i, layer in enumerate(c["layers"]):
        p = "l%d." % i
        y = _layer_norm(x, w(p + "norm1", width), w(p + "norm1.b", width), eps)
        m, q = layer["mixer"]["left"], p + "mix.left."
        nq, nkv, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        wide = {"q": nq * d, "k": nkv * d, "v": nkv * e}
        a = {n: y @ w(q + n, k, width).t() + w(q + n + ".b", k) for n, k in wide.items()}
        grow = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((where + 1) / m["q_temp"]["every"]) + 1)
        a["q"] = _rms(a["q"], w(q + "q.norm", nq * d), eps) * grow[:, None]
        a["k"] = _rms(a["k"], w(q + "k.norm", nkv * d), eps)
        bias = w(q + "rel", BIAS_ROWS, nq)[_distance_rows(max(lens), BIAS_ROWS, m["bias_max"])].t().contiguous()
        o = torch.cat([_causal(a["q"][s:t].view(-1, nq, d), a["k"][s:t].view(-1, nkv, d), a["v"][s:t].view(-1, nkv, e), m["scale"],
                               bias[:, : t - s]) for s, t in zip(starts, starts[1:])])
        o = o * torch.sigmoid(y @ w(q + "g", nq * e, width).t())
        left = o @ w(q + "o", width, nq * e).t() + w(q + "o.b", width)
        m, q = layer["mixer"]["right"], p + "mix.right."
        nh, d, e = m["heads"], m["dim"], m["vdim"]
        qs = (y @ w(q + "q", nh * d, width).t() * d ** -0.5).view(-1, nh, d)
        ks, vs = (y @ w(q + "k", nh * d, width).t()).view(-1, nh, d), (y @ w(q + "v", nh * e, width).t()).view(-1, nh, e)
        z = (y @ w(q + "a1", DECAY_RANK, width).t()) @ w(q + "a2", nh * d, DECAY_RANK).t() + w(q + "a2.b", nh * d)
        keep = (torch.sigmoid(z) ** (1.0 / m["tau"])).view(-1, nh, d)
        o = torch.empty((len(ids), nh, e), dtype=F64, device="cuda")
        # the recurrence, all texts side by side
        state = torch.zeros((len(texts), nh, d, e), dtype=F64, device="cuda")
        for j in range(max(lens)):
            live = [r for r in range(len(lens)) if j < lens[r]]
            rows, r = torch.tensor([starts[r] + j for r in live], device="cuda"), torch.tensor(live, device="cuda")
            s = state[r] * keep[rows][..., None] + ks[rows][..., None] * vs[rows][:, :, None]
            state[r] = s
            o[rows] = (s * qs[rows][..., None]).sum(2)
        o = _rms(o, w(q + "norm", e), eps).reshape(-1, nh * e) * silu(y @ w(q + "g", nh * e, width).t())
        right = o @ w(q + "o", width, nh * e).t()
        x = x + 0.5 * (_rms(left, w(p + "mix.left.out", width), eps) + _rms(right, w(p + "mix.right.out", width), eps))
        y = _layer_norm(x, w(p + "norm2", width), w(p + "norm2.b", width), eps)
        f, q = layer["mlp"], p + "mlp."
        n, ff, shared = f["router"]["experts"], f["expert"]["ff"], f["shared"]["ff"]
        z = y @ w(q + "router", n, width).t() + w(q + "router.b", n)
        top, chosen = torch.topk(z, f["router"]["top"], dim=-1)
        share = torch.zeros_like(z).scatter_(1, chosen, torch.softmax(top, -1))
        add = (silu(y @ w(q + "shared.gate", shared, width).t()) * (y @ w(q + "shared.up", shared, width).t())) @ w(q + "shared.down", width, shared).t()
        for k in range(n):
            rows = share[:, k].nonzero()[:, 0]
            g = silu(y[rows] @ w(q + "e%d.gate" % k, ff, width).t()) * (y[rows] @ w(q + "e%d.up" % k, ff, width).t())
            add.index_add_(0, rows, share[rows, k, None] * (g @ w(q + "e%d.down" % k, width, ff).t()))
        x = x + add
    last = torch.tensor([t - 1 for t in starts[1:]], device="cuda")
    y = _layer_norm(x[last], w("final.norm", width), w("final.norm.b", width), eps)
    z = y @ w("head", c["vocab"], width).t()
    cap = c["logit_softcap"]
    return cap * torch.tanh(z / cap)


def exact(case, seed):
    """What the first pass behind `prepare` returns, in 64 bits; sampled tokens have no such value."""
    if case["kind"] == "sample":
        return None
    tokens = _all_tokens(case, seed)
    if case["kind"] == "prompts":
        texts = tokens
    else:                                                  # the prompt, the token of the pass in `prepare`, and this one's
        texts = [ids[: n + 2] for ids, n in zip(tokens, _lengths(case))] + tokens[case["requests"] :]
    return _exact_nebanex(case, seed, texts) if _is_nebanex(case) else _exact_qwen2(case, seed, texts)
