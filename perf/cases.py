"""The work that a user of this package has it do, as cases that can be timed and compared.

A pass is what an engine does between two looks at its queue: steps of single tokens of requests that are decoding,
prompts that come in (whole, or portions behind what is cached), and whole short requests from the prompt to their last
token.  Tokens are given, so that two runs compute the same thing; logits come back whole, and after the pass the
requests are cut back or closed, so that the next pass does the same again.

A case is a dict:

    design        "qwen3", or one of the other architectures with the layer sizes of a Qwen3 shape
    shape         whose sizes it has; `layers` of them (layers of a kind are alike: a few show them all; four layers of
                  the other designs are one of each of their mechanisms in turn)
    dtype         "bfloat16" or "float32"
    batch         requests that are decoding, each behind about `behind` cached tokens
    prompts       requests that come in, each with `prompt` tokens behind `prompt_behind` cached ones
    steps         steps of one token of every request, after the prompts
    ragged        lengths are spread from 0.4 to 1.6 times the number given; otherwise they are all alike
"""
from __future__ import annotations

import math

import torch

from kipp_amd.config import parse_config, shape_config
from kipp_amd.engine import Engine, Model, StepEntry, model_params
from kipp_amd.runtime import Runtime

PAGE = 16
STEP_TOKENS = 2048          # prompt tokens a step takes, as the scheduler's default
DESIGNS = ("tobinex", "rerizen", "bebulorn", "zivazen", "bipazen", "bavedra")
DEFAULTS = {"design": "qwen3", "shape": "qwen3-4b", "layers": 12, "dtype": "bfloat16", "batch": 0, "behind": 0, "prompts": 0, "prompt": 0,
            "prompt_behind": 0, "steps": 0, "ragged": False}


def _case(**fields):
    return {**DEFAULTS, **fields}


def listed():
    return [
        # one user, one token: the smallest call there is, a chain of launches over weights that are read once
        _case(name="token-1", batch=1, behind=300, steps=1),
        # the headline: eight requests behind prompts of 2,048 tokens
        _case(name="decode-8", batch=8, behind=2048, steps=4),
        # a busy server: many requests of very different lengths, where the cache is most of what is read
        _case(name="decode-64", layers=8, batch=64, behind=1400, steps=2, ragged=True),
        # one prompt of the headline's length
        _case(name="prompt-2048", prompts=1, prompt=2048),
        # a step of continuous batching at the 8B sizes: portions of two prompts beside the tokens of 24 requests
        _case(name="serving", shape="qwen3-8b", layers=6, batch=24, behind=1800, prompts=2, prompt=512, prompt_behind=1500, ragged=True),
        # the 32-bit path: a prompt and its first tokens
        _case(name="float32", layers=3, dtype="float32", prompts=1, prompt=333, steps=2),
        # the other architectures: short and long prompts, few and many requests, then the tokens that follow
        _case(name="tobinex", design="tobinex", layers=4, prompts=1, prompt=1500, steps=4),
        _case(name="rerizen", design="rerizen", layers=4, prompts=8, prompt=150, steps=8, ragged=True),
        _case(name="bebulorn", design="bebulorn", layers=4, prompts=1, prompt=2048),
        _case(name="zivazen", design="zivazen", layers=4, prompts=16, prompt=80, steps=8, ragged=True),
        _case(name="bipazen", design="bipazen", layers=4, prompts=3, prompt=700, steps=4, ragged=True),
        _case(name="bavedra", design="bavedra", layers=4, prompts=1, prompt=1801, steps=6),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Another case of the same ranges: what comes in by its kind, sizes over their logarithms."""
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "serving", "float32"] + list(DESIGNS))
    shape = rng.choice(["qwen3-4b", "qwen3-8b", "qwen3-32b"])
    layers = {"qwen3-4b": rng.choice([6, 8, 12]), "qwen3-8b": rng.choice([4, 6]), "qwen3-32b": rng.choice([2, 3])}[shape]
    if kind == "decode":
        batch = _log_between(rng, 1, 64)
        return _case(shape=shape, layers=layers, batch=batch, behind=_log_between(rng, 30, min(6000, 90000 // batch)), steps=rng.randint(1, 4),
                     ragged=rng.random() < 0.5)
    if kind == "prompt":
        prompt = _log_between(rng, 3, 2048)
        return _case(shape=shape, layers=layers, prompts=1, prompt=prompt, prompt_behind=0 if rng.random() < 0.5 else _log_between(rng, 100, 4000))
    if kind == "serving":
        return _case(shape=shape, layers=layers, batch=_log_between(rng, 2, 32), behind=_log_between(rng, 100, 2000), prompts=rng.randint(1, 3),
                     prompt=_log_between(rng, 20, 420), prompt_behind=_log_between(rng, 16, 2000), ragged=True)
    if kind == "float32":
        return _case(layers=rng.randint(2, 3), dtype="float32", prompts=rng.randint(1, 3), prompt=_log_between(rng, 4, 110), steps=rng.randint(1, 2), ragged=True)
    prompts = _log_between(rng, 1, 24)
    return _case(design=kind, layers=4, prompts=prompts, prompt=_log_between(rng, 6, 1900 // prompts), steps=rng.randint(0, 8), ragged=rng.random() < 0.5)


# ---- models ---------------------------------------------------------------------------------------------------------

def _config(case):
    """The config.json of a case's model."""
    q = shape_config(case["shape"])
    layers = case["layers"]
    if case["design"] == "qwen3":
        q["num_hidden_layers"] = layers
        q["max_position_embeddings"] = 1 << 15
        return q
    width, heads, kv, ff, d = q["hidden_size"], q["num_attention_heads"], q["num_key_value_heads"], q["intermediate_size"], q["head_dim"]
    group = {"heads": heads, "kv_heads": kv, "dim": d, "vdim": d, "scale": d ** -0.5}
    key = 128 if width <= 2560 else 256
    ssd = {"heads": width // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    rglru = {"width": width, "blocks": width // 256, "conv": 4}
    delta = {"heads": 8, "kv_heads": 4, "dim": key, "vdim": width // 8, "conv": 4}
    dense = {"kind": "dense", "ff": ff}
    window = {"size": 1024}
    top = {"architecture": case["design"].capitalize(), "vocab": q["vocab_size"], "width": width, "norm": {"eps": 1e-6}}
    if case["design"] == "tobinex":
        kinds = [("attention", {**group, "mask": None}, dense)]
        top.update(embedding={"scale": 1.0}, postln_alpha=1.0, max_position=8192)
    elif case["design"] == "rerizen":
        attention = {**group, "q_temp": {"coef": 0.1, "every": 512}}
        rot = {"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}
        latent = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 768, "kv_rank": 192, "scale": 192 ** -0.5, "rot": rot, "mask": window}
        mlstm = {"heads": 8, "dim": key, "vdim": width // 8, "gate_cap": 15.0}
        kinds = [("latent_attention", latent, dense), ("attention", attention, dense), ("attention", {**attention, "kv_from": 1}, dense), ("mlstm", mlstm, dense)]
        top.update(streams=2, logit_scale=1.0, max_position=8192)
    elif case["design"] == "bebulorn":
        lightning = {"heads": 8, "dim": key, "vdim": width // 8, "decay": [1.0 - 2.0 ** -(3 + i) for i in range(8)]}
        moe = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}}
        kinds = [("lightning", lightning, dense), ("attention", {**group, "softcap": 30.0, "mask": window}, moe), ("delta", delta, dense), ("lightning", lightning, moe)]
        top.update(norm={"eps": 1e-5}, residual_mult=0.7, loop={"start": 1, "stop": layers, "times": 2})
    elif case["design"] == "zivazen":
        scaling = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}
        attention = {**group, "mask": window, "rot": {"base": 500000.0, "dims": d // 2, "scaling": scaling}, "v_mix": True}
        left = {**group, "mask": window, "rot": {"base": 10000.0, "dims": d // 2}}
        parallel = {"left": left, "right": ssd, "left_scale": 1.25, "right_scale": 0.8}
        moe = {"kind": "moe", "router": {"experts": 32, "top": 4, "groups": {"count": 8, "keep": 4}, "scale": 2.0}, "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}}
        kinds = [("parallel", parallel, dense), ("attention", attention, moe), ("parallel", parallel, moe), ("attention", attention, dense)]
    elif case["design"] == "bipazen":
        latent = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}
        moe = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": ff // 4}}
        kinds = [("mamba2", ssd, moe), ("rglru", rglru, moe), ("rglru", rglru, moe), ("latent_attention", latent, moe)]
        top.update(max_position=8192)
    else:
        left = {**group, "mask": window, "rot": {"base": 10000.0, "dims": d // 2}}
        moe = {"kind": "moe", "router": {"experts": 32, "identity": 8, "top": 4, "groups": {"count": 8, "keep": 4}}, "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}}
        parallel = {"left": left, "right": ssd}
        kinds = [("parallel", parallel, {"kind": "dense", "ff": ff * 3 // 2}), ("delta", delta, moe), ("rglru", rglru, moe), ("parallel", parallel, moe)]
        top.update(embedding={"scale": 1.0}, max_position=8192)
    top["layers"] = [{"type": t, "mixer": dict(m), "mlp": f} for t, m, f in (kinds[i % len(kinds)] for i in range(layers))]
    return top


def _router(config):
    return next((layer["mlp"]["router"] for layer in config.get("layers", ()) if layer["mlp"]["kind"] == "moe"), None)


def _weights(case, seed):
    """Every tensor of the case's model by its file name, as the model's parts declare them, in bfloat16.  Where experts are
    routed, tokens belong to experts as they do in a trained model: an embedding holds the directions of a token's own
    experts, which the routers look for, so that a choice does not hang on the last bit of a rounding."""
    config = _config(case)
    params = model_params(parse_config(config)[1].model_spec())
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.empty(shape, device="cuda").normal_(0.0, 1.0, generator=gen)
    router = _router(config)
    if router is not None:
        choices = router["experts"] + (router.get("identity") or 0)
        directions = normal(choices, config["width"])
    out = {}
    for name, p in params.items():
        how, std = p.init
        t = normal(*p.shape)
        if router is not None and name == "embed":
            own = torch.rand((config["vocab"], choices), device="cuda", generator=gen).topk(router["top"], dim=1).indices
            t += 0.5 * torch.zeros((config["vocab"], choices), device="cuda").scatter_(1, own, 1.0) @ directions
        elif name.endswith(".router"):
            t = 16.0 / config["width"] * directions + 0.001 * t
        elif name.endswith(".correction"):
            t *= 0.5 * std
        elif how == "one_plus_normal":
            t.mul_(std).add_(1.0)
        elif how == "abs_normal":
            t.mul_(std).abs_()
        elif how == "eye_plus_normal":
            t.mul_(std).add_(torch.eye(*p.shape, device="cuda"))
        else:
            t *= std
        out[name] = t.to(torch.bfloat16)
    return out


# ---- requests -------------------------------------------------------------------------------------------------------

def _lengths(case, count, number):
    """`count` lengths: `number` each, or spread from 0.4 to 1.6 times it."""
    if not case["ragged"]:
        return [number] * count
    return [max(1, int(number * (0.4 + 1.2 * ((0.31 + 0.618034 * i) % 1.0)))) for i in range(count)]


def _requests(case, seed):
    """[(name, tokens, cached, prompt)]: the first `cached` tokens are in the cache before the pass, the next `prompt` come
    in one portion, the rest one by one."""
    vocab = shape_config(case["shape"])["vocab_size"]
    gen = torch.Generator().manual_seed(seed + 1)
    sizes = [(f"d{i}", n, 0, max(1, case["steps"])) for i, n in enumerate(_lengths(case, case["batch"], case["behind"]))]
    behind = _lengths(case, case["prompts"], case["prompt_behind"]) if case["prompt_behind"] else [0] * case["prompts"]
    sizes += [(f"p{i}", b, n, case["steps"]) for i, (b, n) in enumerate(zip(behind, _lengths(case, case["prompts"], case["prompt"])))]
    return [(name, torch.randint(0, vocab, (b + n + s,), generator=gen).tolist(), b, n) for name, b, n, s in sizes]


def _steps(case, requests):
    """The steps of a pass: lists of (request index, first token, last token + 1, wanted).  Prompts share a step while they
    fit; requests that are decoding bring a token to the first step of prompts where no steps of single tokens follow."""
    steps, used = [], 0
    coming = [i for i, r in enumerate(requests) if r[3]]
    for i in coming:
        _, _, cached, prompt = requests[i]
        if not steps or used + prompt > STEP_TOKENS:
            steps.append([])
            used = 0
        steps[-1].append((i, cached, cached + prompt, True))
        used += prompt
    decoding = [i for i, r in enumerate(requests) if not r[3]]
    if case["steps"] == 0 and decoding:
        steps[0] = [(i, requests[i][2], requests[i][2] + 1, True) for i in decoding] + steps[0]
    for s in range(case["steps"]):
        steps.append([(i, r[2] + r[3] + s, r[2] + r[3] + s + 1, True) for i, r in enumerate(requests)])
    return steps


def prepare(case, seed):
    """The engine with its model, and the requests that are under way with their tokens in the cache."""
    case = {**DEFAULTS, **case}
    rt = Runtime(case["dtype"])
    model = Model(parse_config(_config(case))[1].model_spec(), rt)
    model.load_tensors(_weights(case, seed))
    requests = _requests(case, seed)
    pages = sum(-(-len(tokens) // PAGE) + 1 for _, tokens, _, _ in requests) + 8
    engine = Engine(model, page_size=PAGE, num_pages=pages, max_requests=len(requests), share_prefixes=False,
                    max_position=max(len(tokens) for _, tokens, _, _ in requests) + PAGE)
    for name, tokens, cached, _ in requests:
        for at in range(0, cached, STEP_TOKENS):
            engine.step([StepEntry(name, tokens[at:min(cached, at + STEP_TOKENS)])])
    steps = [[StepEntry(requests[i][0], requests[i][1][a:b], [b - a - 1] if want else []) for i, a, b, want in step]
             for step in _steps(case, requests)]
    return {"engine": engine, "steps": steps, "after": [(name, cached) for name, _, cached, _ in requests]}


def run(state):
    engine = state["engine"]
    logits = [engine.step(entries) for entries in state["steps"]]
    for name, cached in state["after"]:
        if cached:
            engine.cache.truncate(engine.cache.requests[name], cached)
        else:
            engine.close(name)
    return logits


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def _mixers(config):
    """(kept numbers a token, window, flops a pair, state numbers) of every mixer in run order, parallel ones one by one."""
    if "layers" not in config:
        kv, d, h = config["num_key_value_heads"], config["head_dim"], config["num_attention_heads"]
        return [(2 * kv * d, None, 4 * h * d, 0)] * config["num_hidden_layers"]
    order = list(range(len(config["layers"])))
    loop = config.get("loop")
    if loop:
        order = order[:loop["start"]] + order[loop["start"]:loop["stop"]] * loop["times"] + order[loop["stop"]:]
    out = []
    for i in order:
        m = config["layers"][i]["mixer"]
        for part in ([m["left"], m["right"]] if "left" in m else [m]):
            size = (part.get("mask") or {}).get("size")
            if "kv_rank" in part:
                out.append((part["kv_rank"] + part["rot_dim"], size, 2 * part["heads"] * (2 * part["kv_rank"] + part["rot_dim"]), 0))
            elif "state" in part:
                out.append((0, None, 0, part["heads"] * part["state"] * part["vdim"]))
            elif "width" in part:
                out.append((0, None, 0, part["width"]))
            elif "scale" in part:
                kept = 0 if part.get("kv_from") is not None else part["kv_heads"] * (part["dim"] + part["vdim"])
                out.append((kept, size, 2 * part["heads"] * (part["dim"] + part["vdim"]), 0))
            else:
                out.append((0, None, 0, part["heads"] * part["dim"] * part["vdim"]))
    return out


def work(case):
    """Every step reads each weight that its tokens meet once and the cache of its requests, and writes its tokens' keys and
    values and the logits; a token costs two flops a weight that it meets, and the pairs of its attention."""
    case = {**DEFAULTS, **case}
    config = _config(case)
    spec = parse_config(config)[1].model_spec()
    size = 2 if case["dtype"] == "bfloat16" else 4
    tied = spec.head.tied
    matrices = experts = 0
    for run_ in spec.order:
        prefix = f"model.layers.{run_.layer}." if case["design"] == "qwen3" else f"l{run_.layer}."
        for name, p in model_params(spec).items():
            if name.startswith(prefix) and len(p.shape) >= 2:
                if ".mlp.e" in name:
                    experts += math.prod(p.shape)
                else:
                    matrices += math.prod(p.shape)
    router = _router(config)
    head = spec.vocab_size * spec.hidden_size
    requests = _requests(case, 0)
    nbytes = flops = 0.0
    for step in _steps(case, requests):
        rows = sum(b - a for _, a, b, _ in step)
        wanted = sum(1 for e in step if e[3])
        met, each = 0.0, 0.0
        if router is not None:
            every = router["experts"] + (router.get("identity") or 0)
            each = router["top"] / every
            met = 1.0 - (1.0 - each) ** rows
        nbytes += size * (matrices + met * experts + head + (0 if tied else rows * spec.hidden_size)) + 4 * wanted * spec.vocab_size
        flops += 2.0 * rows * (matrices + each * experts) + 2.0 * wanted * head
        for kept, window, pair, numbers in _mixers(config):
            for _, a, b, _ in step:
                nbytes += size * kept * (min(b, window + b - a) if window else b) + 8 * numbers
                seen = sum(min(t + 1, window) for t in range(a, b)) if window else (b * (b + 1) - a * (a + 1)) / 2
                flops += pair * seen + 6.0 * numbers * (b - a)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Activations between products are rounded to bfloat16: at these depths logits are 0.002 to 0.016 off those in 64 bits
    (5e-6 on the 32-bit path), and another order of the sums moves them by as much again."""
    case = {**DEFAULTS, **case}
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------

def _linear(x, w, b=None):
    y = x @ w.T
    return y if b is None else y + b


def _rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _layer_norm(x, eps, w, b):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu_tanh(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _softplus(x):
    return torch.logaddexp(x, torch.zeros_like(x))


def _frequencies(dims, base, scaling, device):
    """The angles a position adds, and the factor on cosines and sines.  Stretched ones by a ramp over the number of the
    frequency ("fast" and "slow" turns), or by their wavelength ("low" and "high")."""
    i = torch.arange(dims // 2, dtype=torch.float64, device=device)
    f = float(base) ** (-2.0 * i / dims)
    if scaling is None:
        return f, 1.0
    factor, original = scaling["factor"], scaling["original"]
    if "fast" in scaling:
        def at(turns):
            return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        low, high = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), dims - 1)
        ramp = ((i - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0
    share = ((original * f / (2.0 * math.pi) - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0.0, 1.0)
    return (1.0 - share) * f / factor + share * f, 1.0


def _rotate(x, rot, neighbours):
    """x [T, heads, d]: the first `dims` numbers of a head turned by the position, number i with its neighbour or with
    number i + dims / 2.  An angle is formed in float32, position times frequency."""
    freq, factor = _frequencies(rot["dims"], rot["base"], rot.get("scaling"), x.device)
    angle = (torch.arange(x.shape[0], device=x.device).float()[:, None] * freq.float()[None]).double()[:, None]
    cos, sin = torch.cos(angle) * factor, torch.sin(angle) * factor
    part, rest = x[..., :rot["dims"]], x[..., rot["dims"]:]
    if neighbours:
        u, v = part[..., 0::2], part[..., 1::2]
        part = torch.stack([u * cos - v * sin, v * cos + u * sin], dim=-1).flatten(-2)
    else:
        u, v = part.chunk(2, dim=-1)
        part = torch.cat([u * cos - v * sin, v * cos + u * sin], dim=-1)
    return torch.cat([part, rest], dim=-1)


def _attention(q, k, v, scale, window=None, chunk=None, sink=None, cap=None, bias=None, mix=None):
    """q [T, H, d], k [T, G, d], v [T, G, e] -> [T, H, e], causal.  `sink` [H]: a score more in the denominator; `cap`: scores
    through cap tanh(s / cap); `bias` (r1, r2): minus r1 ln(1 + r2 distance); `mix` [H, H]: over the heads after the softmax."""
    t, heads, _ = q.shape
    groups = k.shape[1]
    k, v = (x.permute(1, 0, 2).repeat_interleave(heads // groups, dim=0) for x in (k, v))
    out = []
    block = max(1, int(2e9 // (heads * t * 8)))
    for a in range(0, t, block):
        b = min(t, a + block)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None]
        s = q[a:b].permute(1, 0, 2) @ k[:, :b].transpose(1, 2) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        if bias is not None:
            s = s - bias[0][:, None, None] * torch.log1p(bias[1][:, None, None] * (i - j).clamp(min=0).double())
        seen = j <= i
        if window is not None:
            seen = seen & (i - j < window)
        if chunk is not None:
            seen = seen & (torch.div(i, chunk, rounding_mode="floor") == torch.div(j, chunk, rounding_mode="floor"))
        s = s.masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(heads, b - a, 1)], dim=2)
        p = torch.softmax(s, dim=2)[..., :b]
        if mix is not None:
            p = (mix @ p.reshape(heads, -1)).reshape(p.shape)
        out.append((p @ v[:, :b]).permute(1, 0, 2))
    return torch.cat(out)


def _filter(x, taps, bias=None):
    """Every channel's own causal filter; the last tap weighs the current token."""
    n = taps.shape[1]
    padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    y = sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(n))
    return y if bias is None else y + bias


def _heads(x, n):
    return x.reshape(x.shape[0], n, -1)


def _qwen3(w, c, p, h):
    eps, d = c["rms_norm_eps"], c["head_dim"]
    q, k, v = (_heads(_linear(h, w[p + n + "_proj.weight"]), m) for n, m in (("q", c["num_attention_heads"]), ("k", c["num_key_value_heads"]), ("v", c["num_key_value_heads"])))
    rot = {"dims": d, "base": c["rope_theta"]}
    q, k = (_rotate(_rms(x, eps, w[p + n + "_norm.weight"]), rot, False) for x, n in ((q, "q"), (k, "k")))
    return _linear(_attention(q, k, v, d ** -0.5).flatten(1), w[p + "o_proj.weight"])


def _grouped(w, c, p, m, h, kept):
    """The attention of the other designs; what is not there is left out."""
    eps, design = c["norm"]["eps"], c["architecture"]
    bias = {n: w.get(p + n + ".b") for n in "qkvo"}
    q = _heads(_linear(h, w[p + "q"], bias["q"]), m["heads"])
    size = (m.get("mask") or {}).get("size")
    if design == "Tobinex":
        q = _heads(_rms(q.flatten(1), eps, w[p + "q.norm"]), m["heads"])
        k = _heads(_rms(_linear(h, w[p + "k"]), eps, w[p + "k.norm"]), m["kv_heads"])
        o = _attention(q, k, _heads(_linear(h, w[p + "v"]), m["kv_heads"]), m["scale"], window=size, sink=w[p + "sink"], bias=(w[p + "r1"], w[p + "r2"]), mix=w[p + "talk"])
        return _linear(o.flatten(1) * torch.sigmoid(_linear(h, w[p + "g"])), w[p + "o"])
    if design == "Rerizen":
        t = torch.arange(h.shape[0], device=h.device).double()
        q = _rms(q, eps) * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((t + 1) / m["q_temp"]["every"]) + 1.0))[:, None, None]
        if m.get("kv_from") is None:
            kept["kv"] = _rms(_heads(_linear(h, w[p + "k"], bias["k"]), m["kv_heads"]), eps), _heads(_linear(h, w[p + "v"], bias["v"]), m["kv_heads"])
        return _linear(_attention(q, *kept["kv"], m["scale"]).flatten(1), w[p + "o"])
    k = _heads(_linear(h, w[p + "k"], bias["k"]), m["kv_heads"])
    v = k if p + "v" not in w else _heads(_linear(h, w[p + "v"], bias["v"]), m["kv_heads"])
    if design == "Bebulorn":
        o = _attention(q * w[p + "temp"][:, None], k, _rms(v, eps), m["scale"], window=size, cap=m["softcap"])
        return _linear(o.flatten(1), w[p + "o"])
    if p + "q.norm" in w:
        q, k = _rms(q, eps, w[p + "q.norm"]), _rms(k, eps, w[p + "k.norm"])
    q, k = (_rotate(x, m["rot"], design == "Bavedra") for x in (q, k))
    if m.get("v_mix"):
        if "v" in kept:
            v = (1.0 - w[p + "vmix"]) * v + w[p + "vmix"] * kept["v"]
        else:
            kept["v"] = v
    one = torch.zeros(m["heads"], dtype=torch.float64, device=h.device)
    chunks = design == "Zivazen" and m.get("v_mix")
    o = _attention(q, k, v, m["scale"], window=None if chunks else size, chunk=size if chunks else None, sink=one if chunks or design == "Bavedra" else None)
    return _linear(o.flatten(1), w[p + "o"], bias["o"])


def _latent(w, c, p, m, h, kept):
    eps, heads, d, rank = c["norm"]["eps"], m["heads"], m["dim"], m["kv_rank"]
    stretched = p + "dq" in w
    q = _heads(_linear(_rms(_linear(h, w[p + "dq"]), eps, w[p + "dq.norm"]), w[p + "uq"]) if stretched else _linear(h, w[p + "q"]), heads)
    down = _linear(h, w[p + "dkv"])
    latent, kr = _rms(down[:, :rank], eps, w[p + "dkv.norm"]), _rotate(down[:, None, rank:], m["rot"], stretched)
    q = torch.cat([q[..., :d], _rotate(q[..., d:], m["rot"], stretched)], dim=-1)
    k = torch.cat([_heads(_linear(latent, w[p + "uk"]), heads), kr.expand(-1, heads, -1)], dim=-1)
    o = _attention(q, k, _heads(_linear(latent, w[p + "uv"]), heads), m["scale"], window=(m.get("mask") or {}).get("size"))
    gate = torch.sigmoid(_linear(h, w[p + "g"]))
    return _linear((o * gate[..., None]).flatten(1) if gate.shape[1] == heads else o.flatten(1) * gate, w[p + "o"])


def _mlstm(w, c, p, m, h, kept):
    heads, cap = m["heads"], m["gate_cap"]
    q, k, v = (_heads(_linear(h, w[p + n]), heads) for n in "qkv")
    q = q * m["dim"] ** -0.5
    li, lf = (cap * torch.tanh(_linear(h, w[p + n], w[p + n + ".b"]) / cap) for n in "if")
    lf = -_softplus(-lf)
    s, n, top = h.new_zeros(heads, m["dim"], m["vdim"]), h.new_zeros(heads, m["dim"]), h.new_zeros(heads)
    out = []
    for t in range(h.shape[0]):
        new = torch.maximum(lf[t] + top, li[t])
        keep, take = torch.exp(lf[t] + top - new), torch.exp(li[t] - new)
        s = keep[:, None, None] * s + (take[:, None] * k[t])[:, :, None] * v[t][:, None]
        n, top = keep[:, None] * n + take[:, None] * k[t], new
        below = torch.maximum((n * q[t]).sum(1).abs(), torch.exp(-top)) + 1e-6
        out.append((q[t][:, None] @ s)[:, 0] / below[:, None])
    o = _rms(torch.stack(out), c["norm"]["eps"]).flatten(1) * w[p + "norm"]
    return _linear(o * torch.sigmoid(_linear(h, w[p + "g"])), w[p + "o"])


def _lightning(w, c, p, m, h, kept):
    q, k, v = (_heads(_silu(_linear(h, w[p + n])), m["heads"]) for n in "qkv")
    decay = torch.tensor(m["decay"], dtype=torch.float64, device=h.device)[:, None, None]
    s, out = h.new_zeros(m["heads"], m["dim"], m["vdim"]), []
    for t in range(h.shape[0]):
        s = decay * s + k[t][:, :, None] * v[t][:, None]
        out.append((q[t][:, None] @ s)[:, 0])
    o = _rms(torch.stack(out).flatten(1), c["norm"]["eps"], w[p + "norm"])
    return _linear(o * torch.sigmoid(_linear(h, w[p + "g"])), w[p + "o"])


def _delta(w, c, p, m, h, kept):
    heads, groups = m["heads"], m["kv_heads"]
    q, k, v = (_heads(_silu(_filter(_linear(h, w[p + n]), w[p + n + ".conv"])), g) for n, g in (("q", groups), ("k", groups), ("v", heads)))
    q, k = ((x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // groups, dim=1) for x in (q, k))
    q = q * m["dim"] ** -0.5
    beta = torch.sigmoid(_linear(h, w[p + "b"]))
    g = torch.exp(-torch.exp(w[p + "A_log"]) * _softplus(_linear(h, w[p + "a"]) + w[p + "dt_bias"]))
    s, out = h.new_zeros(heads, m["dim"], m["vdim"]), []
    for t in range(h.shape[0]):
        s = g[t][:, None, None] * s
        u = beta[t][:, None] * (v[t] - (k[t][:, None] @ s)[:, 0])
        s = s + k[t][:, :, None] * u[:, None]
        out.append((q[t][:, None] @ s)[:, 0])
    o = _rms(torch.stack(out), c["norm"]["eps"], w[p + "norm"]).flatten(1)
    return _linear(o * _silu(_linear(h, w[p + "g"])), w[p + "o"])


def _ssd(w, c, p, m, h, kept):
    heads, inner, n = m["heads"], m["heads"] * m["vdim"], m["state"]
    z, xbc, dt = _linear(h, w[p + "in"]).split([inner, inner + 2 * n, heads], dim=1)
    x, b, cc = _silu(_filter(xbc, w[p + "conv"], w[p + "conv.b"])).split([inner, n, n], dim=1)
    x, dt = _heads(x, heads), _softplus(dt + w[p + "dt_bias"])
    decay = torch.exp(-torch.exp(w[p + "A_log"]) * dt)
    s, out = h.new_zeros(heads, n, m["vdim"]), []
    for t in range(h.shape[0]):
        s = decay[t][:, None, None] * s + b[t][None, :, None] * (dt[t][:, None] * x[t])[:, None]
        out.append(cc[t] @ s)
    y = (torch.stack(out) + w[p + "D"][:, None] * x).flatten(1) * _silu(z)
    return _linear(_rms(y, c["norm"]["eps"], w[p + "norm"]), w[p + "o"])


def _rglru(w, c, p, m, h, kept):
    y = _gelu_tanh(_linear(h, w[p + "y"], w[p + "y.b"]))
    u = _filter(_linear(h, w[p + "x"], w[p + "x.b"]), w[p + "conv"], w[p + "conv.b"])
    r, i = (torch.sigmoid(torch.einsum("tbi,boi->tbo", _heads(u, m["blocks"]), w[p + n]) + w[p + n + ".b"]).flatten(1) for n in ("ra", "ri"))
    log_a = -8.0 * r * _softplus(w[p + "lam"])
    a, x = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u
    s, out = torch.zeros_like(u[0]), []
    for t in range(h.shape[0]):
        s = a[t] * s + x[t]
        out.append(s)
    return _linear(torch.stack(out) * y, w[p + "o"])


def _mixer(w, c, layer, p, h, kept):
    m = layer["mixer"]
    if layer["type"] == "parallel":
        left, right = _grouped(w, c, p + "left.", m["left"], h, {}), _ssd(w, c, p + "right.", m["right"], h, kept)
        if c["architecture"] == "Bavedra":
            return 0.5 * (_rms(left, c["norm"]["eps"], w[p + "left.out"]) + _rms(right, c["norm"]["eps"], w[p + "right.out"]))
        return m["left_scale"] * left + m["right_scale"] * right
    kinds = {"attention": _grouped, "latent_attention": _latent, "mlstm": _mlstm, "lightning": _lightning, "delta": _delta, "mamba2": _ssd, "rglru": _rglru}
    return kinds[layer["type"]](w, c, p, m, h, kept)


def _dense(w, design, p, h):
    up = _linear(h, w[p + "up"], w.get(p + "up.b"))
    if design == "Bavedra":
        inner = torch.relu(up) ** 2
    else:
        gate = _linear(h, w[p + "gate"], w.get(p + "gate.b"))
        inner = (torch.relu(gate) if design == "Bebulorn" else _silu(gate)) * up
    return _linear(inner, w[p + "down"], w.get(p + "down.b"))


def _expert(w, design, p, h):
    up = _linear(h, w[p + "up"])
    if design == "Bebulorn":
        inner = 0.5 * up * (1.0 + torch.erf(up / math.sqrt(2.0)))
    elif design == "Zivazen":
        inner = torch.relu(up) ** 2
    else:
        inner = _silu(_linear(h, w[p + "gate"])) * up
    return _linear(inner, w[p + "down"])


def _routed(w, design, p, mlp, h):
    r = mlp["router"]
    z = _linear(h, w[p + "router"])
    s = torch.sigmoid(z) if design in ("Zivazen", "Bipazen") else torch.softmax(z, dim=1)
    rank = s + w[p + "correction"] if p + "correction" in w else s
    if r.get("groups"):
        count, keep = r["groups"]["count"], r["groups"]["keep"]
        of_group = _heads(rank, count).topk(2 if design == "Zivazen" else 1, dim=2).values.sum(2)
        kept = torch.zeros_like(of_group).scatter_(1, of_group.topk(keep, dim=1).indices, 1.0) > 0
        rank = _heads(rank, count).masked_fill(~kept[..., None], -math.inf).flatten(1)
    chosen = rank.topk(r["top"], dim=1).indices
    weight = s.gather(1, chosen)
    if design != "Bipazen":
        weight = weight / (weight.sum(1, keepdim=True) + 1e-20) * (r.get("scale") or 1.0)
    out = torch.zeros_like(h)
    for e in range(z.shape[1]):
        row, place = (chosen == e).nonzero(as_tuple=True)
        if not len(row):
            continue
        a = weight[row, place][:, None]
        if e >= r["experts"]:
            out[row] += a * h[row]
        elif design == "Bipazen":
            out[row] += _expert(w, design, f"{p}e{e}.", a * h[row])
        else:
            out[row] += a * _expert(w, design, f"{p}e{e}.", h[row])
    if mlp.get("shared") is not None:
        shared = _expert(w, design, p + "shared.", h)
        out += torch.sigmoid(_linear(h, w[p + "shared.sg"])) * shared if p + "shared.sg" in w else shared
    return out


def _ff(w, c, layer, p, h):
    return _dense(w, c["architecture"], p, h) if layer["mlp"]["kind"] == "dense" else _routed(w, c["architecture"], p, layer["mlp"], h)


def _logits(c, w, tokens, wanted):
    """float64 logits of the wanted positions of one whole sequence."""
    if "layers" not in c:
        eps = c["rms_norm_eps"]
        x = w["model.embed_tokens.weight"][tokens]
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            x = x + _qwen3(w, c, p + "self_attn.", _rms(x, eps, w[p + "input_layernorm.weight"]))
            h = _rms(x, eps, w[p + "post_attention_layernorm.weight"])
            x = x + _linear(_silu(_linear(h, w[p + "mlp.gate_proj.weight"])) * _linear(h, w[p + "mlp.up_proj.weight"]), w[p + "mlp.down_proj.weight"])
        return _linear(_rms(x[wanted], eps, w["model.norm.weight"]), w["model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"])
    eps, design, layers = c["norm"]["eps"], c["architecture"], c["layers"]
    first = w["embed"][tokens]
    if design == "Zivazen":
        first = _rms(first, eps, w["embed.norm"])
    order = list(range(len(layers)))
    if c.get("loop"):
        order = order[:c["loop"]["start"]] + order[c["loop"]["start"]:c["loop"]["stop"]] * c["loop"]["times"] + order[c["loop"]["stop"]:]
    x, kept, seen = first, {}, set()
    streams = torch.stack([first] * c["streams"]) if design == "Rerizen" else None
    for i in order:
        layer, p = layers[i], f"l{i}."
        if c.get("loop") and i == c["loop"]["start"] and i in seen:
            x = x + first
        seen.add(i)
        if design == "Tobinex":
            x = _rms(c["postln_alpha"] * x + _mixer(w, c, layer, p + "mix.", x, kept), eps, 1.0 + w[p + "norm1"])
            x = _rms(c["postln_alpha"] * x + _ff(w, c, layer, p + "mlp.", x), eps, 1.0 + w[p + "norm2"])
        elif design == "Rerizen":
            for q, f in ((1, lambda h: _mixer(w, c, layer, p + "mix.", h, kept)), (2, lambda h: _ff(w, c, layer, p + "mlp.", h))):
                y = f(_rms(torch.einsum("r,rtw->tw", w[f"{p}hc{q}.in"], streams), eps, w[f"{p}norm{q}"]))
                streams = torch.einsum("rs,rtw->stw", w[f"{p}hc{q}.mix"], streams) + w[f"{p}hc{q}.out"][:, None, None] * y
        elif design == "Bebulorn":
            for n, f in (("norm1", lambda h: _mixer(w, c, layer, p + "mix.", h, kept)), ("norm2", lambda h: _ff(w, c, layer, p + "mlp.", h))):
                y = f(_layer_norm(x, eps, w[p + n], w[p + n + ".b"]))
                x = x + c["residual_mult"] * _layer_norm(y, eps, w[p + n + "b"], w[p + n + "b.b"])
        elif design == "Zivazen":
            h = _rms(x, eps, w[p + "norm1"])
            x = x + _mixer(w, c, layer, p + "mix.", h, kept) + _ff(w, c, layer, p + "mlp.", h)
        else:
            scale = [w.get(p + n, 1.0) for n in ("ls1", "ls2")]
            x = x + scale[0] * _mixer(w, c, layer, p + "mix.", _rms(x, eps, w[p + "norm1"]), kept)
            x = x + scale[1] * _ff(w, c, layer, p + "mlp.", _rms(x, eps, w[p + "norm2"]))
    x = (streams.sum(0) if design == "Rerizen" else x)[wanted]
    if design == "Bebulorn":
        x = _layer_norm(x, eps, w["final.norm"], w["final.norm.b"])
    else:
        x = _rms(x, eps, 1.0 + w["final.norm"] if design == "Tobinex" else w["final.norm"])
    return _linear(x, w["head"] if "head" in w else w["embed"])


def exact(case, seed):
    case = {**DEFAULTS, **case}
    config = _config(case)
    weights = {name: t.double() for name, t in _weights(case, seed).items()}
    requests = _requests(case, seed)
    steps = _steps(case, requests)
    wanted = {i: [] for i in range(len(requests))}
    for step in steps:
        for i, _, b, want in step:
            if want:
                wanted[i].append(b - 1)
    rows = {}
    for i, (_, tokens, _, _) in enumerate(requests):
        logits = _logits(config, weights, torch.tensor(tokens[:wanted[i][-1] + 1], device="cuda"), wanted[i])
        rows.update({(i, at): row for at, row in zip(wanted[i], logits)})
    return [torch.stack([rows[i, b - 1] for i, _, b, want in step if want]) for step in steps]
