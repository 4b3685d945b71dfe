"""The engine's work, as cases that can be timed one by one.

A case is one pass of `EngineCore`: a step of decoding requests, a step of prompts, both mixed, or prompts followed by
a few decoded tokens, with the tokens drawn from the logits on the device, as a serving loop or a trace replay drives it.
Which tokens a request brings is given (seeded ids), so that a pass does not depend on earlier draws.

`listed()` holds the cases, `draw()` makes others of the same ranges, `prepare()` builds the model and fills the caches,
`run()` is one pass, `exact()` what it returns computed in 64 bits by plain torch, `work()` its bytes and operations.
"""

import gc
import math

import torch

from liyab_amd import EngineCore, SamplingParams, StepItem
from liyab_amd.config.registry import config_from_dict
from liyab_amd.sampling import Sampler

# ---------------------------------------------------------------------------------------------------------------
# cases

SIZES = {"small": (12, 768, 12, 3072), "medium": (24, 1024, 16, 4096), "large": (36, 1280, 20, 5120), "xl": (48, 1600, 25, 6400)}
VOCABULARY = 50257
# A case's fields. requests that decode one token each on a cache of `context_low` .. `context_high` tokens; requests that
# bring a portion of a prompt of `prompt_low` .. `prompt_high` tokens, on a cache of `past` tokens; decoded tokens each of
# the latter bring afterwards, a step each (`then`)
FIELDS = {"design": "gpt2", "size": "small", "dtype": "bfloat16", "positions": 1024, "page_size": 16, "invariant": False, "sampling": "greedy",
          "decoding": 0, "context_low": 0, "context_high": 0, "portions": 0, "prompt_low": 0, "prompt_high": 0, "past": 0, "then": 0}


def _case(**fields):
    return dict(FIELDS, **fields)


def listed():
    return [
        # one person's chat: a token at a time, nothing else on the GPU; launches and latency are all of it
        _case(name="small_decode_1", decoding=1, context_low=544, context_high=544),
        # the headline workload: eight requests with prompts of 512 on their way to 1,024 tokens, the default sampling
        _case(name="small_decode_8", decoding=8, context_low=512, context_high=1015, page_size=64, sampling="default"),
        # the same for a service that promises each request the same reply alone and in any batch
        _case(name="small_decode_8_invariant", decoding=8, context_low=512, context_high=1015, invariant=True),
        # a full server: GPT-2 XL's sizes, 64 requests with prompts of 256 on their way to 1,024 tokens
        _case(name="xl_decode_64", size="xl", decoding=64, context_low=256, context_high=1015, page_size=64),
        # prompts of full length, nothing cached: the prefill figure
        _case(name="small_prompts_2x1024", portions=2, prompt_low=1024, prompt_high=1024, page_size=64),
        # the largest step: eight long prompts of odd lengths at GPT-2 XL's sizes (offline scoring, or a burst of requests)
        _case(name="xl_prompts_8x1000", size="xl", portions=8, prompt_low=961, prompt_high=1023),
        # one long document: attention over thousands of keys
        _case(name="small_document_8001", positions=32768, portions=1, prompt_low=8001, prompt_high=8001, page_size=64),
        # continuous batching: portions of ragged prompts beside decoding requests
        _case(name="medium_mixed_16", size="medium", decoding=12, context_low=64, context_high=1011, portions=4, prompt_low=127, prompt_high=256, past=256),
        # the 32-bit path: a few prompts and short replies, as a conformance run or an evaluation has them
        _case(name="small_float32", dtype="float32", portions=4, prompt_low=100, prompt_high=511, then=8),
        # the other designs: prompts and short replies
        _case(name="lafanex_small", design="lafanex", portions=4, prompt_low=180, prompt_high=640, then=8),
        _case(name="lolulorn_small", design="lolulorn", portions=4, prompt_low=180, prompt_high=640, then=8),
        _case(name="bokulix_small", design="bokulix", portions=4, prompt_low=180, prompt_high=640, then=8),
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["decode", "decode", "prompts", "prompts", "mixed", "float32", "design", "design"])
    page = rng.choice([16, 64])
    if kind == "decode":
        size = rng.choice(["small", "small", "medium", "large", "xl"])
        low = rng.randint(16, 600)
        return _case(size=size, decoding=_log_uniform(rng, 1, 64), context_low=low, context_high=rng.randint(low, 1015), page_size=page,
                     invariant=size == "small" and rng.random() < 0.25, sampling=rng.choice(["greedy", "default"]))
    if kind == "prompts":
        size = rng.choice(["small", "medium", "large", "xl"])
        if size == "small" and rng.random() < 0.3:
            n = _log_uniform(rng, 1024, 8001)
            return _case(positions=32768, portions=1, prompt_low=n, prompt_high=n, page_size=page)
        high = _log_uniform(rng, 16, 1023)
        return _case(size=size, portions=_log_uniform(rng, 1, 7), prompt_low=rng.randint(max(2, high // 3), high), prompt_high=high, page_size=page)
    if kind == "mixed":
        low = rng.randint(16, 600)
        high = _log_uniform(rng, 16, 256)
        return _case(size=rng.choice(["small", "medium", "large"]), decoding=_log_uniform(rng, 1, 48), context_low=low, context_high=rng.randint(low, 1011),
                     portions=rng.randint(1, 6), prompt_low=rng.randint(max(2, high // 3), high), prompt_high=high, past=rng.choice([0, 256, 512]), page_size=page)
    high = _log_uniform(rng, 16, 511 if kind == "float32" else 640)
    design = {"dtype": "float32"} if kind == "float32" else {"design": rng.choice(["lafanex", "lolulorn", "bokulix"]), "size": rng.choice(["small", "small", "medium"])}
    return _case(portions=_log_uniform(rng, 1, 8 if kind == "design" else 4), prompt_low=rng.randint(max(2, high // 3), high), prompt_high=high,
                 then=rng.randint(1, 8), page_size=page, **design)


def _spread(low, high, n):
    """`n` lengths from `low` to `high`, both among them, in no order."""
    return [low + (high - low) * ((i * 5 + n - 1) % n if math.gcd(5, n) == 1 else n - 1 - i) // max(n - 1, 1) for i in range(n)]


def _requests(case):
    """(cached, new) tokens of every request of the pass, the decoding ones first."""
    return ([(c, 1) for c in _spread(case["context_low"], case["context_high"], case["decoding"])]
            + [(case["past"], n) for n in _spread(case["prompt_low"], case["prompt_high"], case["portions"])])


# ---------------------------------------------------------------------------------------------------------------
# models

def _config(case):
    L, d, H, F = SIZES[case["size"]]
    P, hd, dense = case["positions"], d // H, max(64, F * 2 // 3 // 64 * 64)
    if case["design"] == "gpt2":
        return {"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2", "n_layer": L, "n_embd": d, "n_head": H, "n_inner": F, "vocab_size": VOCABULARY,
                "n_positions": P, "layer_norm_epsilon": 1e-5, "activation_function": "gelu_new", "tie_word_embeddings": True}
    common = {"vocab": VOCABULARY, "width": d, "norm": {"eps": 1e-5}, "max_positions": P}
    if case["design"] == "bokulix":  # two of eight experts, together as wide as GPT-2's feed-forward; cached rows of 128
        layer = {"type": "latent_attention", "mixer": {"heads": H, "dim": hd, "vdim": hd, "kv_rank": 128, "scale": hd ** -0.5, "mask": {"size": P}},
                 "mlp": {"kind": "moe", "expert": {"ff": F // 2}, "router": {"experts": 8, "top": 2}}}
        return dict(common, architecture="Bokulix", canon={"taps": 4}, layers=[layer] * L)
    gated = {"kind": "dense", "ff": dense}
    attention = {"heads": H, "kv_heads": H, "dim": hd, "vdim": hd, "scale": hd ** -0.5}
    if case["design"] == "lolulorn":  # a gated delta rule, gated linear attention over experts, attention under a window
        moe = {"kind": "moe", "expert": {"ff": F // 4}, "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}}}
        window = dict(attention, mask={"size": P // 2, "keep_first": 4}, rot={"dims": hd, "base": 10000.0, "scaling": {"factor": 4.0}})
        layers = []
        for i in range(L):
            if i % 3 == 0:
                layers.append({"type": "delta", "mixer": {"heads": H, "kv_heads": H // 2 if H % 2 == 0 else H, "dim": hd, "vdim": hd, "conv": 4}, "mlp": gated})
            elif i % 3 == 1:
                layers.append({"type": "gla", "mixer": {"heads": H, "dim": hd, "vdim": hd, "tau": 16.0, "decay_rank": 16}, "mlp": moe})
            else:
                layers.append({"type": "attention", "mixer": dict(window, **({"kv_from": i - 3} if i % 6 == 5 else {})), "mlp": gated})
        return dict(common, architecture="Lolulorn", embedding={"scale": 1.0}, layers=layers)
    # lafanex: two residual streams; attention, a selective scan, attention over experts
    expert = {"ff": F // 4, "limit": 7.0}
    moe = {"kind": "moe", "expert": expert, "router": {"experts": 8, "top": 2, "identity": 2, "scale": 2.5}, "shared": expert}
    turned = dict(attention, rot={"dims": hd, "base": 10000.0})
    kinds = [{"type": "attention", "mixer": turned, "mlp": gated},
             {"type": "mamba1", "mixer": {"inner": 2 * d, "state": 16, "dt_rank": max(8, d // 16), "conv": 4}, "mlp": gated},
             {"type": "attention", "mixer": turned, "mlp": moe}]
    return dict(common, architecture="Lafanex", streams=2, layers=[kinds[i % 3] for i in range(L)])


class _Asked:
    """Stands where a store of weights stands while a model is built, and notes the tensors it is asked for."""

    def __init__(self):
        self.device, self.compute_dtype = torch.device("meta"), torch.float32
        self.sources = {}  # name -> (stored shape, role, distribution)

    def has(self, src):
        return src.required

    def fetch(self, src, shape, role, keep=True):
        if not src.required:
            return None
        shape = tuple(int(s) for s in shape)
        stored = shape[::-1] if src.layout == "in_out" else shape
        self.sources[src.name] = (stored, role, src.init)
        return torch.empty(shape, device="meta")

    def fetch_joined(self, srcs, shapes, role, how="rows"):
        parts = [self.fetch(s, shape, role) for s, shape in zip(srcs, shapes)]
        return torch.cat(parts) if how == "rows" else torch.stack(parts)

    def derived(self, key, make):
        return make()


def _sources(plan):
    from liyab_amd.models.decoder import DecoderModel

    asked = _Asked()
    DecoderModel(plan, asked, torch.float32)
    return asked.sources


def _tensors(case, plan, seed):
    """The model's weights by name, on the GPU: matrices and tables in the path's type, vectors in 32 bits. The designs with
    routers get token rows that outweigh a single layer's update, as trained ones do: with a stream made of updates alone, a
    choice of experts that flips within a rounding changes the logits by half their size, and nothing could be compared."""
    out = {}
    generator = torch.Generator(device="cuda:0")
    for i, (name, (shape, role, init)) in enumerate(sorted(_sources(plan).items())):
        generator.manual_seed(seed * 100003 + i)
        t = torch.randn(shape, generator=generator, device="cuda:0").mul_(init.std if init else 0.02).add_(init.mean if init else 0.0)
        if name == "embed":
            t.mul_(16.0 / init.std)
        out[name] = t.to(torch.bfloat16) if role in ("matrix", "table") and case["dtype"] == "bfloat16" else t
    return out


def _ids(case, seed):
    """A request's token ids, as many as it holds at the end of a pass: arrays on the host."""
    generator = torch.Generator().manual_seed(seed + 17)
    return [torch.randint(0, VOCABULARY, (cached + new + case["then"],), generator=generator).numpy() for cached, new in _requests(case)]


_SAMPLING = {"greedy": SamplingParams(temperature=0.0), "default": SamplingParams(seed=1)}


def prepare(case, seed):
    """The engine with its model, every request's cache filled up to the pass, and the items that the pass brings."""
    plan = config_from_dict(_config(case)).plan()
    requests, ids = _requests(case), _ids(case, seed)
    pages = sum(-(-(cached + new + case["then"]) // case["page_size"]) for cached, new in requests) + 4
    gc.collect()
    core = EngineCore.from_plan(plan, _tensors(case, plan, seed), dtype=case["dtype"], page_size=case["page_size"], num_pages=pages,
                                max_requests=max(2, len(requests)), context_length=case["positions"], batch_invariant=case["invariant"])
    kept = [r for r, (cached, _) in enumerate(requests) if cached]
    new = [r for r, (cached, _) in enumerate(requests) if not cached]
    for r in kept:
        core.open(r)
    fill, room = [], 2048  # the caches, in steps of up to 2,048 tokens
    for r in kept:
        at = 0
        while at < requests[r][0]:
            n = min(room, requests[r][0] - at)
            fill.append(StepItem(r, ids[r][at:at + n]))
            at, room = at + n, room - n
            if not room:
                core.step(fill)
                fill, room = [], 2048
    if fill:
        core.step(fill)
    steps = [[StepItem(r, ids[r][c:c + n], [n - 1]) for r, (c, n) in enumerate(requests)]]
    for k in range(case["then"]):
        steps.append([StepItem(r, ids[r][c + n + k:c + n + k + 1], [0]) for r, (c, n) in enumerate(requests)])
    return {"core": core, "sampler": Sampler(core.device), "steps": steps, "new": new, "back": [(r, requests[r][0]) for r in kept],
            "params": [_SAMPLING[case["sampling"]]] * len(requests), "seeds": [1000 + r for r in range(len(requests))]}


def run(state):
    """One pass: new requests are opened, every step runs and its tokens are drawn; afterwards new requests are closed and
    the others rolled back to where they were. Logits and tokens of every step."""
    core, sampler, rows = state["core"], state["sampler"], len(state["seeds"])
    for r in state["new"]:
        core.open(r)
    out = {}
    for k, items in enumerate(state["steps"]):
        logits = core.step(items)
        tokens = sampler.sample_on_device(logits, state["params"], state["seeds"], [k] * rows)
        more = len(state["steps"]) > 1  # (a step's logits and tokens are valid until the next one's)
        out[f"logits_{k}"] = logits.clone() if more else logits
        if rows > 1:  # (a single row's token is drawn too: alone, one that flips within the rounding would be all of the output)
            out[f"tokens_{k}"] = tokens.clone() if more else tokens
    for r in state["new"]:
        core.close(r)
    for r, length in state["back"]:
        core.truncate(r, length)
    return out


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    """Matrices read once a step (of a layer's experts as many as its tokens can choose), cached keys and values and states read,
    new ones written, logits written; products, attention's scores and weighted sums, recurrences token by token."""
    config, requests = _config(case), _requests(case)
    plan = config_from_dict(config).plan()
    elt = 2 if case["dtype"] == "bfloat16" else 4
    sources = _sources(plan)
    steps = [requests] + [[(c + n + k, 1) for c, n in requests] for k in range(case["then"])]
    total_bytes = total_flops = 0.0
    layers = config.get("layers") or [{"type": "attention", "mixer": {"heads": config["n_head"], "kv_heads": config["n_head"], "dim": config["n_embd"] // config["n_head"],
                                                                      "vdim": config["n_embd"] // config["n_head"]}}] * config["n_layer"]
    for step in steps:
        tokens = sum(n for _, n in step)
        pairs = sum(n * c + n * (n + 1) / 2 for c, n in step)
        for name, (shape, role, _) in sources.items():
            size = math.prod(shape)
            if name in ("wte.weight", "head.weight", "head", "embed", "wpe.weight", "pos"):
                continue
            if role == "vector":
                total_bytes += size * 4
                continue
            expert = ".mlp.e" in name
            if expert:
                r = next(l["mlp"]["router"] for l in layers if (l.get("mlp") or {}).get("kind") == "moe")
                share, chosen = r["top"] / (r["experts"] + r.get("identity", 0)), r["experts"]
                total_bytes += size * elt * min(1.0, tokens * r["top"] / chosen)
                total_flops += 2.0 * size * tokens * share
            else:
                total_bytes += size * elt
                total_flops += 2.0 * size * tokens
        width = config.get("width") or config["n_embd"]
        total_bytes += VOCABULARY * width * elt + tokens * width * elt + len(step) * VOCABULARY * 4  # the head, the tokens' rows, the logits
        total_flops += 2.0 * VOCABULARY * width * len(step)
        for layer in layers:
            m = layer["mixer"]
            if layer["type"] == "attention":
                total_bytes += sum(c + n for c, n in step) * m["kv_heads"] * (m["dim"] + m["vdim"]) * elt
                total_flops += 2.0 * pairs * m["heads"] * (m["dim"] + m["vdim"])
            elif layer["type"] == "latent_attention":
                total_bytes += sum(c + n for c, n in step) * m["kv_rank"] * elt
                total_flops += 2.0 * pairs * m["heads"] * 2 * m["dim"]
            elif layer["type"] == "mamba1":
                total_bytes += len(step) * 2 * m["inner"] * m["state"] * 4
                total_flops += 7.0 * tokens * m["inner"] * m["state"]
            else:
                total_bytes += len(step) * 2 * m["heads"] * m["dim"] * m["vdim"] * 4
                total_flops += tokens * m["heads"] * m["dim"] * m["vdim"] * (8.0 if layer["type"] == "delta" else 5.0)
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """About four times what is seen between the path and `exact`: 4e-7 in 32 bits, 3.8e-3 in bfloat16; designs with routers
    show 2e-3 to 1e-2, and 3e-2 where a token's choice of experts flips within the rounding. Tokens: a row whose largest
    logits lie within the rounding may draw another one."""
    one_row = 1.0 / max(2, case["decoding"] + case["portions"])
    if case["dtype"] == "float32":
        return {"rel": 2e-6, "differ": 0.1}
    return {"rel": 1.5e-2 if case["design"] == "gpt2" else 1e-1, "differ": max(0.3, one_row)}


# ---------------------------------------------------------------------------------------------------------------
# the same in 64 bits: whole sequences, no cache, no carried state

def _gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def _silu(z):
    return z * torch.sigmoid(z)


def _unit(v, eps):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _centred(v, w, b, eps):
    return torch.nn.functional.layer_norm(v, v.shape[-1:], w, b, eps)


def _turn(v, rot):
    """Pairs (2i, 2i + 1) of the first rot.dims entries of every head turned by position * base^(-2i / dims) / factor."""
    dims, n = rot["dims"], v.shape[0]
    f = rot["base"] ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=v.device) / dims) / (rot.get("scaling") or {"factor": 1.0})["factor"]
    a = torch.arange(n, dtype=torch.float64, device=v.device)[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    out = v.clone()
    out[..., 0:dims:2] = v[..., 0:dims:2] * c - v[..., 1:dims:2] * s
    out[..., 1:dims:2] = v[..., 1:dims:2] * c + v[..., 0:dims:2] * s
    return out


def _attend(q, k, v, scale, mask=None, one=False):
    """q, k, v [n, heads, dim], as many key heads as query heads; `one`: one is added to the softmax's denominator."""
    n = q.shape[0]
    out = torch.empty(n, q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    j = torch.arange(n, device=q.device)
    for at in range(0, n, 1024):
        i = j[at:at + 1024, None]
        seen = j[None, :] <= i
        if mask:
            seen = seen & ((i - j[None, :] < mask["size"]) | (j[None, :] < mask.get("keep_first", 0)))
        for h in range(q.shape[1]):
            s = (q[at:at + 1024, h] @ k[:, h].t()) * scale
            s = s.masked_fill(~seen, -math.inf)
            if one:
                s = torch.cat([s, torch.zeros_like(s[:, :1])], dim=1)
            out[at:at + 1024, h] = torch.softmax(s, dim=-1)[:, :n] @ v[:, h]
    return out.reshape(n, -1)


def _convolve(x, w, b=None):
    """x [n, channels], w [channels, taps] (last column: the current row), zeros before the first row."""
    n, taps = x.shape[0], w.shape[1]
    padded = torch.cat([torch.zeros(taps - 1, x.shape[1], dtype=x.dtype, device=x.device), x])
    out = sum(w[:, j] * padded[j:j + n] for j in range(taps))
    return out if b is None else out + b


def _experts(h, chosen, weights, count, expert):
    out = torch.zeros_like(h)
    for e in range(count):
        row, place = (chosen == e).nonzero(as_tuple=True)
        if len(row):
            out.index_add_(0, row, weights[row, place, None] * expert(h[row], e))
    return out


def _exact_gpt2(config, t, ids):
    n, H = len(ids), config["n_head"]
    x = t["wte.weight"][ids] + t["wpe.weight"][:n]
    for i in range(config["n_layer"]):
        def part(name, y):
            return y @ t[f"h.{i}.{name}.weight"] + t[f"h.{i}.{name}.bias"]

        q, k, v = part("attn.c_attn", _centred(x, t[f"h.{i}.ln_1.weight"], t[f"h.{i}.ln_1.bias"], 1e-5)).reshape(n, 3, H, -1).unbind(1)
        x = x + part("attn.c_proj", _attend(q, k, v, q.shape[-1] ** -0.5))
        x = x + part("mlp.c_proj", _gelu(part("mlp.c_fc", _centred(x, t[f"h.{i}.ln_2.weight"], t[f"h.{i}.ln_2.bias"], 1e-5))))
    return lambda rows: _centred(x[rows], t["ln_f.weight"], t["ln_f.bias"], 1e-5) @ t["wte.weight"].t()


def _exact_bokulix(config, t, ids):
    n, eps = len(ids), config["norm"]["eps"]
    x = t["embed"][ids] + t["pos"][:n]
    for i, layer in enumerate(config["layers"]):
        m, r = layer["mixer"], layer["mlp"]["router"]
        w = {k[len(f"l{i}."):]: v for k, v in t.items() if k.startswith(f"l{i}.")}
        u = x + _convolve(x, w["canon1"])
        c = _unit(u @ w["mix.dkv"].t(), eps) * w["mix.dkv.norm"]
        q, k, v = (y.reshape(n, m["heads"], -1) for y in (u @ w["mix.q"].t(), c @ w["mix.uk"].t(), c @ w["mix.uv"].t()))
        y = (_attend(q, k, v, m["scale"], m["mask"]) * torch.sigmoid(u @ w["mix.g"].t())) @ w["mix.o"].t()
        x = x + _unit(y * torch.sigmoid(x @ w["rg1"].t() + w["rg1.b"]), eps) * w["norm1"]
        best = torch.topk(x @ w["mlp.router"].t() + w["mlp.router.b"], r["top"], dim=-1)
        y = _experts(x, best.indices, torch.softmax(best.values, dim=-1), r["experts"], lambda h, e: (
            _silu(h @ w[f"mlp.e{e}.gate"].t()) * (h @ w[f"mlp.e{e}.up"].t())) @ w[f"mlp.e{e}.down"].t())
        x = x + _unit(y * torch.sigmoid(x @ w["rg2"].t() + w["rg2.b"]), eps) * w["norm2"]
    return lambda rows: (_unit(x[rows], eps) * t["final.norm"]) @ t["head"].t()


def _exact_lolulorn(config, t, ids):
    n, eps, kept = len(ids), config["norm"]["eps"], {}
    x = t["embed"][ids] * config["embedding"]["scale"]
    for i, layer in enumerate(config["layers"]):
        m, f = layer["mixer"], layer["mlp"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        w = {k[len(f"l{i}."):]: v for k, v in t.items() if k.startswith(f"l{i}.")}

        def of(name):
            return x @ w["mix." + name].t()

        if layer["type"] == "attention":
            if m.get("kv_from") is None:
                kept[i] = (_turn((_unit(of("k"), eps) * w["mix.k.norm"]).reshape(n, H, D), m["rot"]), of("v").reshape(n, H, V))
            q = _turn((_unit(of("q"), eps) * w["mix.q.norm"]).reshape(n, H, D), m["rot"])
            y = _attend(q, *kept[i if m.get("kv_from") is None else m["kv_from"]], m["scale"], m["mask"]) @ w["mix.o"].t()
        else:
            if layer["type"] == "delta":
                G = m["kv_heads"]
                q, k, v = (_silu(_convolve(of(c), w[f"mix.{c}.conv"])) for c in "qkv")
                q, k = (y.reshape(n, G, D) / torch.sqrt((y.reshape(n, G, D) ** 2).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
                q, k, v = q.repeat_interleave(H // G, 1) * D ** -0.5, k.repeat_interleave(H // G, 1), v.reshape(n, H, V)
                rate = torch.sigmoid(of("b"))
                decay = torch.exp(-torch.exp(w["mix.A_log"]) * torch.nn.functional.softplus(of("a") + w["mix.dt_bias"]))[..., None].expand(n, H, D)
            else:
                q, k, v = of("q").reshape(n, H, D) * D ** -0.5, of("k").reshape(n, H, D), of("v").reshape(n, H, V)
                decay = torch.exp(torch.nn.functional.logsigmoid(of("a1") @ w["mix.a2"].t() + w["mix.a2.b"]) / m["tau"]).reshape(n, H, D)
            S, o = torch.zeros(H, D, V, dtype=x.dtype, device=x.device), []
            for p in range(n):
                S = decay[p][..., None] * S
                new = v[p] if layer["type"] == "gla" else rate[p][:, None] * (v[p] - (k[p][..., None] * S).sum(1))
                S = S + k[p][..., None] * new[:, None]
                o.append((q[p][..., None] * S).sum(1))
            y = ((_unit(torch.stack(o), eps) * w["mix.norm"]).reshape(n, -1) * _silu(of("g"))) @ w["mix.o"].t()
        x = x + _centred(y, w["norm1"], w["norm1.b"], eps)
        if f["kind"] == "dense":
            y = (_gelu(x @ w["mlp.gate"].t()) * (x @ w["mlp.up"].t())) @ w["mlp.down"].t()
        else:
            r = f["router"]
            E, G = r["experts"], r["groups"]["count"]
            s = torch.sigmoid(x @ w["mlp.router"].t())
            c = s + w["mlp.correction"]
            stay = torch.topk(torch.topk(c.reshape(n, G, E // G), 2, dim=-1).values.sum(-1), r["groups"]["keep"], dim=-1).indices
            allowed = torch.zeros(n, G, dtype=torch.bool, device=x.device).scatter_(1, stay, True).repeat_interleave(E // G, 1)
            chosen = torch.topk(c.masked_fill(~allowed, -math.inf), r["top"], dim=-1).indices
            y = _experts(x, chosen, s.gather(1, chosen), E, lambda h, e: (
                _silu(h @ w[f"mlp.e{e}.gate"].t()) * (h @ w[f"mlp.e{e}.up"].t())) @ w[f"mlp.e{e}.down"].t())
        x = x + _centred(y, w["norm2"], w["norm2.b"], eps)
    return lambda rows: _centred(x[rows], t["final.norm"], t["final.norm.b"], eps) @ t["head"].t()


def _exact_lafanex(config, t, ids):
    n, eps = len(ids), config["norm"]["eps"]
    X = t["embed"][ids].expand(config["streams"], -1, -1)

    for i, layer in enumerate(config["layers"]):
        m, f = layer["mixer"], layer["mlp"]
        w = {k[len(f"l{i}."):]: v for k, v in t.items() if k.startswith(f"l{i}.")}

        def mix(x):
            h = _unit(x, eps) * (1.0 + w["norm1"])
            if layer["type"] == "attention":
                q, k, v = ((h @ w["mix." + c].t()).reshape(n, m["heads"], -1) for c in "qkv")
                return _attend(_unit(_turn(q, m["rot"]), eps), _unit(_turn(k, m["rot"]), eps), v, m["scale"], one=True) @ w["mix.o"].t()
            N, rank = m["state"], m["dt_rank"]
            x, z = (h @ w["mix.in"].t()).split(m["inner"], dim=-1)
            x = _silu(_convolve(x, w["mix.conv"], w["mix.conv.b"]))
            d, B, C = (x @ w["mix.x"].t()).split([rank, N, N], dim=-1)
            d = torch.nn.functional.softplus(d @ w["mix.dt"].t() + w["mix.dt.b"])
            A, S, y = -torch.exp(w["mix.A_log"]), 0.0, []
            for p in range(n):
                S = torch.exp(d[p][:, None] * A) * S + (d[p] * x[p])[:, None] * B[p]
                y.append(S @ C[p])
            return ((torch.stack(y) + w["mix.D"] * x) * _silu(z)) @ w["mix.o"].t()

        def unit(h, name, limit):
            g, u = (h @ w[f"mlp.{name}gate"].t()).clamp(max=limit), (h @ w[f"mlp.{name}up"].t()).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[f"mlp.{name}down"].t()

        def feed(x):
            h = _unit(x, eps) * (1.0 + w["norm2"])
            if f["kind"] == "dense":
                return (_gelu(h @ w["mlp.gate"].t()) * (h @ w["mlp.up"].t())) @ w["mlp.down"].t()
            r = f["router"]
            p = torch.softmax(h @ w["mlp.router"].t(), dim=-1)
            chosen = torch.topk(p + w["mlp.correction"], r["top"], dim=-1).indices
            out = _experts(h, chosen, r["scale"] * p.gather(1, chosen), r["experts"] + r["identity"],
                           lambda g, e: g if e >= r["experts"] else unit(g, f"e{e}.", f["expert"]["limit"]))
            return out + torch.sigmoid(h @ w["mlp.shared.sg"].t()) * unit(h, "shared.", f["shared"]["limit"])

        for q, sublayer in ((1, mix), (2, feed)):
            y = sublayer(torch.einsum("s,snd->nd", w[f"hc{q}.in"], X))
            X = torch.einsum("st,snd->tnd", w[f"hc{q}.mix"], X) + w[f"hc{q}.out"][:, None, None] * y
    return lambda rows: (_unit(X.sum(0)[rows], eps) * (1.0 + t["final.norm"])) @ t["embed"].t()


def exact(case, seed):
    """What `run` returns, from whole sequences in float64. Tokens drawn with a temperature have no such value."""
    config = _config(case)
    t = {name: v.double() for name, v in _tensors(case, config_from_dict(config).plan(), seed).items()}
    forward = {"gpt2": _exact_gpt2, "bokulix": _exact_bokulix, "lolulorn": _exact_lolulorn, "lafanex": _exact_lafanex}[case["design"]]
    rows = []
    for (cached, new), ids in zip(_requests(case), _ids(case, seed)):
        logits = forward(config, t, torch.from_numpy(ids).to("cuda:0"))
        rows.append(logits(slice(cached + new - 1, None)))
    out = {}
    for k in range(case["then"] + 1):
        logits = torch.stack([r[k] for r in rows])
        out[f"logits_{k}"] = logits
        if len(rows) > 1:
            out[f"tokens_{k}"] = logits.argmax(-1).to(torch.int32) if case["sampling"] == "greedy" else None
    return out
