"""The work that a user has this engine do, as cases to be timed and compared.

A case is one pass of the step function (`ModelRunner.step`, which `LLM.generate`, the command line and
`bin/trace_run` all run) over a batch of single tokens and prompt portions whose earlier tokens are in the
cache, or a whole `LLMEngine.generate` of many short requests.  The layer sizes are those of the published
Qwen2.5 models that the package ships as presets and, for Bevovik (routed experts, latent attention, gated
linear attention, gated recurrence), those that bench.py gives it beside them.  Weights are random, as
everywhere in this package's benchmark: N(0, 0.02), norms around one.

Keys of a case: `task` "step" or "generate"; `model` "qwen2" or "bevovik"; `size`; `dtype`;
  step:     `decodes` sequences with `low` to `high` tokens in the cache take one token each, beside
            `prompts` portions of `first` to `last` tokens that begin at position `start`;
  generate: `requests` prompts of `first` to `last` tokens, up to `new` generated tokens each, every second
            one drawn with temperature and top_p.
"""

from __future__ import annotations

import hashlib
import math

import torch

from shrike_amd import LLMEngine, SamplingParams
from shrike_amd.cache import CacheManager
from shrike_amd.config import EngineConfig
from shrike_amd.config.presets import load_preset
from shrike_amd.engine.runner import ModelRunner, StepEntry
from shrike_amd.engine.runtime import Runtime
from shrike_amd.models import DecoderModel, bevovik, qwen2

PAGE = 16  # tokens of a cache page, the engine's default
DEVICE = "cuda:0"
CLASSES = 64  # token classes that Bevovik's routers tell apart
CLASS_SIZE = 4.0


def _step(name, model, size, dtype, decodes=0, low=0, high=0, prompts=0, first=0, last=0, start=0):
    case = dict(task="step", model=model, size=size, dtype=dtype, decodes=decodes, low=low, high=high,
                prompts=prompts, first=first, last=last, start=start)
    return dict(name=name, **case) if name else case


def _generate(name, size, requests, first, last, new):
    case = dict(task="generate", model="qwen2", size=size, dtype="bfloat16", requests=requests, first=first, last=last,
                new=new)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # one user's next token from a small model: a few hundred short kernels, bound by launches and latency
        _step("decode 0.5b b1", "qwen2", "0.5b", "bfloat16", decodes=1, low=333, high=333),
        # the headline of bench.py: eight users behind 2,048-token prompts
        _step("decode 7b b8", "qwen2", "7b", "bfloat16", decodes=8, low=2048, high=2076),
        # a busy server: 64 users of all lengths
        _step("decode 7b b64 ragged", "qwen2", "7b", "bfloat16", decodes=64, low=61, high=1203),
        # a whole prompt in one step: the time to the first token
        _step("prompt 7b 2048", "qwen2", "7b", "bfloat16", prompts=1, first=2048, last=2048),
        # several short prompts of odd lengths admitted together
        _step("prompts 0.5b ragged", "qwen2", "0.5b", "bfloat16", prompts=5, first=37, last=411),
        # a portion of the default token budget far into a long document
        _step("portion 7b at 12000", "qwen2", "7b", "bfloat16", prompts=1, first=512, last=512, start=12001),
        # running users beside a newcomer's prompt portion under the default budget of 512 tokens
        _step("mixed 14b 32+480", "qwen2", "14b", "bfloat16", decodes=32, low=123, high=456, prompts=1, first=480, last=480),
        # the true float32 mode: a prompt, and a few users' next tokens
        _step("prompt 0.5b float32", "qwen2", "0.5b", "float32", prompts=1, first=509, last=509),
        _step("decode 0.5b b4 float32", "qwen2", "0.5b", "float32", decodes=4, low=201, high=402),
        # routed experts, latent attention and recurrent mixers: a prompt, and eight users' next tokens
        _step("prompt bevovik 1501", "bevovik", "7b", "bfloat16", prompts=1, first=1501, last=1501),
        _step("decode bevovik b8", "bevovik", "7b", "bfloat16", decodes=8, low=700, high=1001),
        # an offline run through generate(): admission, prompt portions beside decodes, sampling, the host's part
        _generate("generate 0.5b 32", "0.5b", requests=32, first=24, last=72, new=32),
    ]


def _between(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "portion", "mixed", "float32", "bevovik", "bevovik", "generate"])
    if kind == "generate":
        first = _between(rng, 8, 60)
        return _generate(None, "0.5b", _between(rng, 1, 48), first, first + rng.randint(0, 60), _between(rng, 4, 40))
    size, dtype, model = rng.choice(["0.5b", "7b", "7b", "14b"]), "bfloat16", "qwen2"
    if kind == "float32":
        size, dtype, kind = "0.5b", "float32", rng.choice(["decode", "prompt"])
    if kind == "bevovik":
        size, model, kind = rng.choice(["0.5b", "7b"]), "bevovik", rng.choice(["decode", "prompt"])
    if kind == "decode":
        batch = _between(rng, 1, 64 if dtype == "bfloat16" and model == "qwen2" else 16)
        high = _between(rng, 40, {"qwen2": 3000, "bevovik": 1500}[model] if batch <= 12 else 1100)
        return _step(None, model, size, dtype, decodes=batch, low=rng.randint(1 + high // 9, high), high=high)
    if kind == "prompt":
        total = _between(rng, 24, 2048 if size != "14b" and dtype == "bfloat16" else 700)
        count = rng.choice([1, 1, 1, 2, 5])
        last = max(1, total // count)
        return _step(None, model, size, dtype, prompts=count, first=rng.randint(1 + last // 3, last), last=last)
    if kind == "portion":
        n = _between(rng, 64, 1024 if size != "14b" else 512)
        return _step(None, model, size, dtype, prompts=1, first=n, last=n, start=_between(rng, 500, 14000 if size != "14b" else 5000))
    n, high = _between(rng, 40, 480), _between(rng, 40, 1000)
    return _step(None, model, size, dtype, decodes=_between(rng, 2, 32), low=rng.randint(1 + high // 9, high), high=high,
                 prompts=1, first=n, last=n)


# ------------------------------------------------------------------------------ models and weights


def _spread_over(low, high, count):
    """`count` whole numbers from low to high at even distances."""
    return [low + (high - low) * i // max(1, count - 1) for i in range(count)]


def _sequences(case):
    """[(tokens in the cache, new tokens)] of a step's sequences."""
    out = [(n, 1) for n in _spread_over(case["low"], case["high"], case["decodes"])]
    return out + [(case["start"], n) for n in _spread_over(case["first"], case["last"], case["prompts"])]


def _qwen2_raw(case):
    raw = load_preset("qwen2.5-" + case["size"])
    if case["task"] == "generate":
        raw["tie_word_embeddings"] = False  # see _weight: the output matrix is a permutation of the embedding
    return raw


def _bevovik_raw(case):
    """Bevovik with the layer sizes of a Qwen2.5 preset, as bench.py's --bevovik makes it."""
    q = load_preset("qwen2.5-" + case["size"])
    h, d, inter = q["hidden_size"], q["head_dim"], q["intermediate_size"]

    def up64(x):
        return max(64, -(-int(x) // 64) * 64)

    latent = dict(heads=q["num_attention_heads"], dim=d, rot_dim=d // 2, vdim=d, q_rank=up64(3 * h / 8),
                  kv_rank=min(up64(h / 8), 512), scale=(1.5 * d) ** -0.5,
                  rot=dict(base=10000.0, dims=d // 2, scaling=dict(factor=4.0, original=4096.0, fast=32.0, slow=1.0)))
    gla = dict(heads=max(1, h // 256), dim=128, vdim=256, tau=16.0, decay_rank=16)
    rec = dict(width=h, blocks=h // (256 if h % 256 == 0 else 128), conv=4)
    mlp = dict(kind="moe", expert=dict(ff=max(64, inter // 4 // 64 * 64), limit=7.0),
               router=dict(experts=8, top=2, identity=2, scale=2.0, groups=dict(count=2, keep=1)),
               shared=dict(ff=up64(inter / 2), limit=7.0))
    kinds = [("rglru", rec), ("latent_attention", latent), ("gla", gla)]
    layers = [dict(type=kinds[i % 3][0], mixer=kinds[i % 3][1], mlp=mlp) for i in range(q["num_hidden_layers"])]
    return dict(architecture="Bevovik", vocab=q["vocab_size"], width=h, norm=dict(eps=q["rms_norm_eps"]), layers=layers,
                torch_dtype="bfloat16")


def _number(seed, text):
    return int.from_bytes(hashlib.sha256(f"{seed}:{text}".encode()).digest()[:7], "little")


def _generator(seed, text, device=DEVICE):
    return torch.Generator(device=device).manual_seed(_number(seed, text))


def _stays_float32(name):
    """Vectors that enter float32 arithmetic are held so; matrices are held in the compute dtype."""
    return "norm" in name or name.endswith((".b", ".bias", ".ls1", ".ls2", ".conv", ".lam", ".a2", ".correction"))


def _weight(case, seed, name, shape):
    """A tensor of the weight file.  In "generate" cases the output matrix is the embedding with its rows
    permuted, so that every next token is a permutation of the last, by a wide margin: sequences of tokens
    that rounding does not change."""
    permuted = case["task"] == "generate" and name == "lm_head.weight"
    gen = _generator(seed, "model.embed_tokens.weight" if permuted else name)
    t = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(0.0, 1.0, generator=gen)
    if permuted:
        t = t[torch.randperm(shape[0], generator=_generator(seed, "permutation"), device=DEVICE)]
    elif name in ("model.embed_tokens.weight", "embed"):
        pass
    elif name.endswith(("o_proj.weight", "down_proj.weight")):
        t.mul_(0.02 * (2 * load_preset("qwen2.5-" + case["size"])["num_hidden_layers"]) ** -0.5)
    elif name.endswith((".ls1", ".ls2")):
        t.mul_(0.1).add_(1.0).mul_((2 * load_preset("qwen2.5-" + case["size"])["num_hidden_layers"]) ** -0.5)
    elif "norm" in name:
        t.mul_(0.1).add_(1.0)
    elif name.endswith(".conv"):
        t.mul_(0.3)
        t[:, -1] += 1.0
    elif name.endswith(".lam"):
        t.mul_(1.5).sub_(5.0)
    elif name.endswith(".router"):
        # A router reads the elements of the stream that name the token's class (the embedding sets them, no
        # layer's output reaches them): experts are loaded unevenly, as in use, and no choice is a close call.
        t[:, :CLASSES] *= 2.0 / CLASS_SIZE
        t[:, CLASSES:] = 0.0
    else:
        t.mul_(0.02)
    if case["model"] == "bevovik" and name == "embed":
        ids = torch.arange(shape[0], device=DEVICE)
        t[:, :CLASSES] = 0.0
        t[ids, ids % CLASSES] = CLASS_SIZE
    elif case["model"] == "bevovik" and name.endswith((".norm1", ".norm2")):
        t[:CLASSES] = 0.0
    return t if _stays_float32(name) else t.to(getattr(torch, case["dtype"]))


def _model(case, seed):
    if case["model"] == "bevovik":
        spec = bevovik.build_spec(bevovik.BevovikConfig.from_dict(_bevovik_raw(case)))
    else:
        spec = qwen2.build_spec(qwen2.Qwen2Config.from_dict(_qwen2_raw(case)))
    model, runtime = DecoderModel(spec), Runtime(DEVICE, getattr(torch, case["dtype"]))
    model.load({p.name: _weight(case, seed, p.name, p.drawn_shape()) for p in model.params() if not p.optional},
               runtime)
    return model, runtime


def _vocab(case):
    return load_preset("qwen2.5-" + case["size"])["vocab_size"]


def _tokens(case, seed):
    """One list of token ids per sequence of the step, or per request."""
    if case["task"] == "generate":
        lengths = _spread_over(case["first"], case["last"], case["requests"])
    else:
        lengths = [have + new for have, new in _sequences(case)]
    ids = torch.randint(_vocab(case), (sum(lengths),), generator=_generator(seed, "tokens", "cpu")).tolist()
    out = []
    for n in lengths:
        out.append(ids[:n])
        ids = ids[n:]
    return out


# ------------------------------------------------------------------------------ a pass


def prepare(case, seed):
    """Weights on the device, a cache, and the tokens before the step already in it."""
    model, runtime = _model(case, seed)
    tokens = _tokens(case, seed)
    if case["task"] == "generate":
        pages = sum(-(-(len(t) + case["new"]) // PAGE) + 1 for t in tokens)
        engine = LLMEngine(None, EngineConfig(block_size=PAGE, num_kv_blocks=pages, enable_prefix_caching=False,
                                              dtype=case["dtype"], seed=seed), model=model, runtime=runtime)
        new = _spread_over(max(1, case["new"] // 2), case["new"], len(tokens))
        sampling = [SamplingParams(max_new_tokens=n, ignore_eos=True, temperature=0.8 * (i % 2), top_p=0.95 if i % 2 else 1.0)
                    for i, n in enumerate(new)]
        return {"engine": engine, "prompts": tokens, "sampling": sampling}
    pages = sum(-(-len(t) // PAGE) for t in tokens)
    cache = CacheManager(model.cache_specs(), PAGE, pages, max_slots=len(tokens), enable_prefix_caching=False)
    cache.allocate(runtime.dtype, runtime.device)
    runner = ModelRunner(model, cache, runtime)
    entries, ahead = [], []
    for (have, _new), ids in zip(_sequences(case), tokens):
        seq = cache.new_sequence()
        cache.append(seq, 0, len(ids))
        entries.append(StepEntry(seq, ids[have:], have, [len(ids) - have - 1]))
        ahead += [(seq, ids[at : min(have, at + 2048)], at) for at in range(0, have, 2048)]
    while ahead:  # earlier tokens, up to 4,096 a step
        batch, rest, room = [], [], 4096
        for seq, ids, at in ahead:
            if len(ids) <= room and all(seq is not e.cache for e in batch) and all(seq is not r[0] for r in rest):
                batch.append(StepEntry(seq, ids, at, []))
                room -= len(ids)
            else:
                rest.append((seq, ids, at))
        runner.step(batch)
        ahead = rest
    return {"runner": runner, "entries": entries}


def run(state):
    if "engine" in state:
        out = state["engine"].generate(state["prompts"], state["sampling"], chat=False)
        return torch.tensor([token for tokens in out for token in tokens])
    return state["runner"].step(state["entries"])


# ------------------------------------------------------------------------------ what a pass cannot do without


def work(case):
    elem = 2 if case["dtype"] == "bfloat16" else 4
    q = load_preset("qwen2.5-" + case["size"])
    h, layers, vocab = q["hidden_size"], q["num_hidden_layers"], q["vocab_size"]
    if case["task"] == "generate":
        prompts = _spread_over(case["first"], case["last"], case["requests"])
        new = _spread_over(max(1, case["new"] // 2), case["new"], case["requests"])
        sequences = [(0, p + n - 1) for p, n in zip(prompts, new)]
        wanted, passes = sum(new), case["new"]
    else:
        sequences, passes = _sequences(case), 1
        wanted = len(sequences)
    tokens = sum(n for _, n in sequences)
    pairs = sum(n * have + n * (n + 1) // 2 for have, n in sequences)  # (query, key) pairs
    cached = sum(have for have, _ in sequences) + tokens
    if case["model"] == "bevovik":
        raw = _bevovik_raw(case)
        rec, lat, gla = (raw["layers"][i]["mixer"] for i in range(3))
        counts = [sum(layer["type"] == kind for layer in raw["layers"]) for kind in ("rglru", "latent_attention", "gla")]
        H, row = lat["heads"], lat["kv_rank"] + lat["rot_dim"]
        mixers = [3 * h * rec["width"] + 2 * rec["width"] ** 2 // rec["blocks"],
                  (lat["q_rank"] + row) * h + H * (lat["dim"] + lat["rot_dim"]) * lat["q_rank"]
                  + 2 * H * lat["dim"] * lat["kv_rank"] + H * lat["vdim"] * h,
                  (2 * 128 + 3 * 256) * gla["heads"] * h + 16 * (h + 128 * gla["heads"])]
        mlp = raw["layers"][0]["mlp"]
        ff, shared, router = mlp["expert"]["ff"], mlp["shared"]["ff"], mlp["router"]
        outputs = router["experts"] + router["identity"]
        picked = router["top"] * router["experts"] / outputs  # of a token's choices, those with matrices
        touched = router["experts"] * (1.0 - (1.0 - picked / router["experts"]) ** tokens)
        fixed = sum(c * m for c, m in zip(counts, mixers)) + layers * (outputs * h + 3 * h * shared)
        state = 2 * 4 * len(sequences) * (counts[0] * 4 * rec["width"] + counts[2] * gla["heads"] * 128 * 256)
        nbytes = elem * (fixed + layers * touched * 3 * h * ff + vocab * h + counts[1] * cached * row) + state
        flops = 2.0 * tokens * (fixed + layers * picked * 3 * h * ff) + 2.0 * wanted * vocab * h
        flops += 2.0 * pairs * counts[1] * H * (lat["dim"] + lat["rot_dim"] + lat["vdim"]) + 4.0 * tokens * counts[2] * gla["heads"] * 128 * 256
    else:
        H, KV, d = q["num_attention_heads"], q["num_key_value_heads"], q["head_dim"]
        matrices = layers * (2 * (H + KV) * d * h + 3 * h * q["intermediate_size"])
        nbytes = elem * (passes * (matrices + vocab * h) + layers * cached * 2 * KV * d)
        flops = 2.0 * tokens * matrices + 2.0 * wanted * vocab * h + 4.0 * pairs * layers * H * d
    return {"bytes": float(nbytes + 4 * wanted * vocab), "flops": float(flops)}


def tolerance(case):
    """About four times the distance from 64-bit logits that was measured: 6.5e-7 in float32, in bfloat16 0.0018
    for the 0.5B sizes, 0.0053 for 7B, 0.008 for 14B and 0.0036 for Bevovik (the deeper, the more)."""
    if case["task"] == "generate":
        return "exact"  # see _weight: rounding does not reach the tokens
    if case["dtype"] == "float32":
        rel = 3e-6
    elif case["model"] == "bevovik":
        rel = 0.015
    else:
        rel = {"0.5b": 0.008, "7b": 0.02, "14b": 0.03}[case["size"]]
    return {"rel": rel, "max": 10 * rel}


# ------------------------------------------------------------------------------ the same in 64 bits


def exact(case, seed):
    """Logits at the wanted places from the whole sequences, in float64, without a cache."""
    if case["task"] == "generate":
        return None
    rows, where, at = [], [], 0
    tokens = _tokens(case, seed)
    for ids in tokens:
        where.append((at, at + len(ids)))
        at += len(ids)
        rows.append(at - 1)
    ids = torch.tensor([i for t in tokens for i in t], device=DEVICE)

    def w(name, *shape):
        return _weight(case, seed, name, shape).double()

    with torch.no_grad():
        return (_exact_bevovik if case["model"] == "bevovik" else _exact_qwen2)(case, seed, w, ids, where, rows)


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _embedded(case, seed, name, ids, width):
    return _weight(case, seed, name, (_vocab(case), width))[ids].double()


def _causal(q, k, v, scale):
    """softmax(q k^T scale) v for queries [heads, n, d] that share the keys [n, d] and values [n, e]."""
    heads, n, d = q.shape
    out = torch.empty(heads, n, v.shape[1], dtype=q.dtype, device=q.device)
    for lo in range(0, n, 1024):
        hi = min(n, lo + 1024)
        s = (q[:, lo:hi].reshape(-1, d) @ k[:hi].T).view(heads, hi - lo, hi).mul_(scale)
        s.masked_fill_(torch.ones(hi - lo, hi, dtype=torch.bool, device=q.device).triu_(lo + 1), float("-inf"))
        out[:, lo:hi] = (torch.softmax(s, -1).view(-1, hi) @ v[:hi]).view(heads, hi - lo, -1)
    return out


def _exact_qwen2(case, seed, w, ids, where, rows):
    q = _qwen2_raw(case)
    h, inter, eps, vocab = q["hidden_size"], q["intermediate_size"], q["rms_norm_eps"], q["vocab_size"]
    H, KV, d = q["num_attention_heads"], q["num_key_value_heads"], q["head_dim"]
    x = _embedded(case, seed, "model.embed_tokens.weight", ids, h)
    positions = torch.cat([torch.arange(b - a, device=DEVICE) for a, b in where]).double()
    rates = q["rope_theta"] ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEVICE) / d)
    cos, sin = torch.cos(positions[:, None] * rates), torch.sin(positions[:, None] * rates)

    def turn(t):
        a, b = t[..., : d // 2], t[..., d // 2 :]
        return torch.cat([a * cos[:, None] - b * sin[:, None], b * cos[:, None] + a * sin[:, None]], -1)

    for i in range(q["num_hidden_layers"]):
        p = f"model.layers.{i}."
        y = _rms(x, eps) * w(p + "input_layernorm.weight", h)
        a = p + "self_attn."
        qs = turn((y @ w(a + "q_proj.weight", H * d, h).T + w(a + "q_proj.bias", H * d)).view(-1, H, d))
        ks = turn((y @ w(a + "k_proj.weight", KV * d, h).T + w(a + "k_proj.bias", KV * d)).view(-1, KV, d))
        vs = (y @ w(a + "v_proj.weight", KV * d, h).T + w(a + "v_proj.bias", KV * d)).view(-1, KV, d)
        out, per = torch.empty_like(qs), H // KV
        for lo, hi in where:
            for g in range(KV):
                mine = slice(g * per, (g + 1) * per)
                out[lo:hi, mine] = _causal(qs[lo:hi, mine].transpose(0, 1), ks[lo:hi, g], vs[lo:hi, g], d**-0.5).transpose(0, 1)
        x = x + out.view(-1, H * d) @ w(a + "o_proj.weight", h, H * d).T
        if i == q["num_hidden_layers"] - 1:
            x = x[rows]
        y = _rms(x, eps) * w(p + "post_attention_layernorm.weight", h)
        g = y @ w(p + "mlp.gate_proj.weight", inter, h).T
        g = g * torch.sigmoid(g)
        g *= y @ w(p + "mlp.up_proj.weight", inter, h).T
        x = x + g @ w(p + "mlp.down_proj.weight", h, inter).T
    head = "model.embed_tokens.weight" if q["tie_word_embeddings"] else "lm_head.weight"
    return (_rms(x, eps) * w("model.norm.weight", h)) @ w(head, vocab, h).T


def _exact_bevovik(case, seed, w, ids, where, rows):
    raw = _bevovik_raw(case)
    h, eps = raw["width"], raw["norm"]["eps"]
    x = _embedded(case, seed, "embed", ids, h)
    longest = max(b - a for a, b in where)
    # sequences side by side, each from its first token, for what goes token by token
    place = torch.stack([torch.arange(longest, device=DEVICE).clamp(max=b - a - 1) + a for a, b in where])
    inside = torch.stack([torch.arange(longest, device=DEVICE) < b - a for a, b in where])

    def joined(t):  # [sequences, longest, ...] -> [tokens, ...]
        return t[inside]

    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}.mix", layer["mixer"]
        if layer["type"] == "rglru":
            width, blocks = m["width"], m["blocks"]
            part = width // blocks
            y = torch.nn.functional.gelu(x @ w(p + ".y", width, h).T + w(p + ".y.b", width), approximate="tanh")
            u = (x @ w(p + ".x", width, h).T + w(p + ".x.b", width))[place]
            taps, c = w(p + ".conv", width, m["conv"]), w(p + ".conv.b", width).expand_as(u).clone()
            for k in range(m["conv"]):
                c[:, k:] += taps[:, m["conv"] - 1 - k] * u[:, : longest - k]
            r, g = (torch.empty_like(c) for _ in range(2))
            for out, name in ((r, ".ra"), (g, ".ri")):
                mat, bias = w(p + name, blocks, part, part), w(p + name + ".b", blocks, part)
                for b in range(blocks):
                    at = slice(b * part, (b + 1) * part)
                    out[..., at] = torch.sigmoid(c[..., at] @ mat[b].T + bias[b])
            log_a = -8.0 * r * torch.nn.functional.softplus(w(p + ".lam", width))
            a, add = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * g * c
            S, read = torch.zeros_like(add[:, 0]), torch.empty_like(add)
            for t in range(longest):
                S = torch.addcmul(add[:, t], a[:, t], S)
                read[:, t] = S
            y = (joined(read) * y) @ w(p + ".o", h, width).T
        elif layer["type"] == "latent_attention":
            H, D, R, V, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            cq = _rms(x @ w(p + ".dq", m["q_rank"], h).T, eps) * w(p + ".dq.norm", m["q_rank"])
            qs = (cq @ w(p + ".uq", H * (D + R), m["q_rank"]).T).view(-1, H, D + R)
            down = x @ w(p + ".dkv", rank + R, h).T
            c = _rms(down[:, :rank], eps) * w(p + ".dkv.norm", rank)
            turn = _turner(m["rot"], torch.cat([torch.arange(b - a, device=DEVICE) for a, b in where]))
            q_rot, k_rot = turn(qs[..., D:]), turn(down[:, None, rank:])[:, 0]
            ks, vs = (c @ w(p + ".uk", H * D, rank).T).view(-1, H, D), (c @ w(p + ".uv", H * V, rank).T).view(-1, H, V)
            out = torch.empty(x.shape[0], H, V, dtype=x.dtype, device=DEVICE)
            qs = torch.cat([qs[..., :D], q_rot], -1)
            for lo, hi in where:
                for head in range(H):
                    k = torch.cat([ks[lo:hi, head], k_rot[lo:hi]], -1)
                    out[lo:hi, head] = _causal(qs[lo:hi, head][None], k, vs[lo:hi, head], m["scale"])[0]
            y = out.view(-1, H * V) @ w(p + ".o", h, H * V).T
        else:
            H, D, V = m["heads"], m["dim"], m["vdim"]
            qs = (x @ w(p + ".q", H * D, h).T).view(-1, H, D)[place] * D**-0.5
            ks, vs = (x @ w(p + ".k", H * D, h).T).view(-1, H, D)[place], (x @ w(p + ".v", H * V, h).T).view(-1, H, V)[place]
            z = (x @ w(p + ".a1", m["decay_rank"], h).T) @ w(p + ".a2", H * D, m["decay_rank"]).T + w(p + ".a2.b", H * D)
            alpha = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(-1, H, D)[place]
            S = torch.zeros(len(where), H, D, V, dtype=x.dtype, device=DEVICE)
            read = torch.empty(len(where), longest, H, V, dtype=x.dtype, device=DEVICE)
            for t in range(longest):
                S.mul_(alpha[:, t, :, :, None]).addcmul_(ks[:, t, :, :, None], vs[:, t, :, None, :])
                read[:, t] = (S * qs[:, t, :, :, None]).sum(2)
            g = x @ w(p + ".g", H * V, h).T
            y = (_rms(joined(read), eps) * w(p + ".norm", V)).view(-1, H * V)
            y = (y * g * torch.sigmoid(g)) @ w(p + ".o", h, H * V).T
        x = x + _rms(y, eps) * w(f"l{i}.norm1", h) * w(f"l{i}.ls1", h)
        if i == len(raw["layers"]) - 1:
            x = x[rows]
        x = x + _rms(_exact_mixture(w, f"l{i}.mlp", layer["mlp"], x), eps) * w(f"l{i}.norm2", h) * w(f"l{i}.ls2", h)
    return (_rms(x, eps) * w("final.norm", h)) @ w("head", raw["vocab"], h).T


def _turner(rot, positions):
    """Turns neighbouring pairs of the last axis at rates that YaRN stretches."""
    base, dims, sc = rot["base"], rot["dims"], rot["scaling"]

    def place(turns):
        return dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    first, last = max(math.floor(place(sc["fast"])), 0), min(math.ceil(place(sc["slow"])), dims - 1)
    number = torch.arange(dims // 2, dtype=torch.float64, device=DEVICE)
    share = ((number - first) / max(last - first, 0.001)).clamp(0.0, 1.0)
    rates = base ** (-2.0 * number / dims)
    angle = positions.double()[:, None] * (rates / sc["factor"] * share + rates * (1.0 - share))
    size = 0.1 * math.log(sc["factor"]) + 1.0
    cos, sin = (torch.cos(angle) * size)[:, None], (torch.sin(angle) * size)[:, None]

    def turn(t):
        u, v = t[..., 0::2], t[..., 1::2]
        return torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2)

    return turn


def _exact_mixture(w, p, m, x):
    h, r, ff = x.shape[1], m["router"], m["expert"]["ff"]

    def expert(t, prefix, ff, limit):
        g = (t @ w(prefix + ".gate", ff, h).T).clamp(max=limit)
        u = (t @ w(prefix + ".up", ff, h).T).clamp(min=-limit, max=limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(prefix + ".down", h, ff).T

    outputs, count = r["experts"] + r["identity"], r["groups"]["count"]
    scores = torch.softmax(x @ w(p + ".router", outputs, h).T, -1)
    choice = scores + w(p + ".correction", outputs)
    best = choice.view(-1, count, outputs // count).amax(-1)
    keep = torch.zeros_like(best).scatter_(1, best.topk(r["groups"]["keep"], 1).indices, 1.0)
    choice = choice.masked_fill(keep.repeat_interleave(outputs // count, 1) == 0, float("-inf"))
    chosen = choice.topk(r["top"], 1).indices
    weights = scores.gather(1, chosen)
    weights = weights / (weights.sum(-1, keepdim=True) + 1e-20) * r["scale"]
    out = expert(x, p + ".shared", m["shared"]["ff"], m["shared"]["limit"])
    for e in range(outputs):
        at, slot = (chosen == e).nonzero(as_tuple=True)
        if at.numel():
            y = x[at] if e >= r["experts"] else expert(x[at], f"{p}.e{e}", ff, m["expert"]["limit"])
            out.index_add_(0, at, y * weights[at, slot, None])
    return out
