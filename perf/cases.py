"""The calls that this engine is measured at, with inputs, outputs, work and 64-bit answers.

A case names a model of the sizes that the repository's benchmark uses, a numeric type, and one of three calls of the
step function:

    prompt   a batch of prompts that have just arrived: slots taken, one step over all tokens, the logits of each
             prompt's last token, slots given back
    decode   one more token for each of a batch of sequences that the cache holds (the step is then wound back, so that
             every pass finds the same context)
    serve    a batch of prompts and then `new` more tokens each, one step a token (models with recurrent layers, whose
             state cannot be wound back); the tokens are given, so that a pass does not depend on near ties of logits

Weights are random (N(0, 0.02)), token ids uniform: nothing is downloaded.  `tokens` is the longest sequence of the
batch, `shortest` the shortest, the others lie between.
"""
import math
import random
import re

import torch

from cpmcu_amd import Engine, EngineOptions, StepEntry, get_architecture
from cpmcu_amd.weights import random_tensors

DEVICE = "cuda:0"
VOCAB = 73448
CHUNK = 2048                     # tokens a forward pass, the engine's own default


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    case = lambda name, model, call, batch, tokens, shortest=0, new=0, layers=0, dtype="bfloat16": {
        "name": name, "model": model, "call": call, "batch": batch, "tokens": tokens, "shortest": shortest or tokens,
        "new": new, "layers": layers, "dtype": dtype}
    return [
        # one user talks to the small model: the smallest call, a chain of short launches
        case("0.5b decode 1", "small", "decode", 1, 300),
        # a busy server of the small model: the benchmark's 64 unequal sequences
        case("0.5b decode 64 unequal", "small", "decode", 64, 2048, 128),
        # the 32-bit engine, which results are checked against: two odd prompts
        case("0.5b fp32 prompt 2", "small", "prompt", 2, 333, 190, dtype="float32"),
        # the benchmark's own decode step: 8 sequences at 4,096 tokens, all 32 layers
        case("8b decode 8", "8b", "decode", 8, 4096),
        # the benchmark's own prompt (half of the layers)
        case("8b prompt 2048", "8b", "prompt", 1, 2048, layers=16),
        # a long document through block-sparse attention, chunk by chunk (a quarter of the layers)
        case("8b sparse prompt", "8b sparse", "prompt", 1, 20011, layers=8),
        # the other architectures, four layers of a real model's sizes each: a whole pass of prompts ...
        case("duvulix prompt 2048", "duvulix", "prompt", 1, 2048),
        case("gumodra prompts ragged", "gumodra", "prompt", 5, 613, 77),
        case("sagedra prompt 1500", "sagedra", "prompt", 1, 1500),
        case("pemalorn prompt 2048", "pemalorn", "prompt", 1, 2048),
        # ... and requests answered in a batch: prompts, then a token a step
        case("nelutar serve 8", "nelutar", "serve", 8, 200, 60, new=24),
        case("tirizen serve 24", "tirizen", "serve", 24, 300, 40, new=16),
    ]


def draw(rng):
    over = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    model = rng.choice(["small", "small", "8b", "8b sparse", "duvulix", "gumodra", "sagedra", "nelutar", "pemalorn", "tirizen"])
    own = model in ("small", "8b", "8b sparse")
    call = rng.choice(["prompt", "decode" if own else "serve"])
    c = {"model": model, "call": call, "new": 0, "layers": 8 if model.startswith("8b") else 0, "dtype": "bfloat16"}
    if model == "8b sparse":
        c["batch"], c["tokens"] = (1, over(4096, 20000)) if call == "prompt" else (rng.randint(1, 3), over(8500, 20000))
    elif call == "prompt":
        c["batch"] = over(1, 8)
        c["tokens"] = over(3, 4096 if c["batch"] <= 2 else 8192 // c["batch"])
        if model == "small" and rng.random() < 0.3:
            c["dtype"], c["tokens"] = "float32", min(c["tokens"], 700 // c["batch"])
    elif call == "decode":
        c["batch"] = over(1, 64)
        c["tokens"] = over(20, min(8192, 65536 // c["batch"]))
        if model == "small" and rng.random() < 0.2:
            c["dtype"], c["tokens"] = "float32", min(c["tokens"], 500)
            c["batch"] = min(c["batch"], 4)
    else:
        c["batch"], c["tokens"], c["new"] = over(1, 32), over(8, 400), rng.randint(6, 24)
    c["shortest"] = over(max(1, c["tokens"] // 16), c["tokens"])
    return c


def lengths(case):
    """The batch's lengths, spread between the shortest and the longest in a mixed order."""
    B, lo, hi = case["batch"], case["shortest"], case["tokens"]
    return [hi] if B == 1 else [lo + (hi - lo) * ((5 * i + 3) % B) // (B - 1) for i in range(B)]


# ---------------------------------------------------------------------------------------------------- the models
def _minicpm(layers, hidden, heads, dim, ff, tied, sparse=None):
    factors = [1.0 + 3.0 * ((11 * i) % (dim // 2)) / (dim // 2) for i in range(dim // 2)]
    raw = {"architectures": ["MiniCPMForCausalLM"], "model_type": "minicpm", "num_hidden_layers": layers,
           "hidden_size": hidden, "num_attention_heads": heads, "num_key_value_heads": 2, "head_dim": dim,
           "intermediate_size": ff, "vocab_size": VOCAB, "rms_norm_eps": 1e-6, "rope_theta": 10000.0,
           "max_position_embeddings": 32768,
           "rope_scaling": {"rope_type": "longrope", "short_factor": factors, "long_factor": factors,
                            "original_max_position_embeddings": 32768},
           "scale_emb": 12, "dim_model_base": 256, "scale_depth": 1.4, "tie_word_embeddings": tied,
           "hidden_act": "silu", "torch_dtype": "bfloat16"}
    return dict(raw, sparse_config=sparse) if sparse else raw


def _decays():
    return [1.0 - 2.0 ** (-5.0 - 3.0 * h / 31.0) for h in range(32)]


def _duvulix():
    latent = {"heads": 32, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
              "rot": {"base": 500000.0, "dims": 64}}
    attn = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
            "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}},
            "mask": {"size": 2048}}
    mamba = {"heads": 128, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    mlp = {"kind": "dense", "ff": 16384}
    return {"architecture": "Duvulix", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6}, "layers": [
        {"type": "latent_attention", "mixer": dict(latent), "mlp": mlp}, {"type": "attention", "mixer": attn, "mlp": mlp},
        {"type": "mamba2", "mixer": mamba, "mlp": mlp}, {"type": "latent_attention", "mixer": dict(latent, kv_from=0), "mlp": mlp}]}


def _gumodra():
    attn = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
            "rot": {"base": 500000.0, "dims": 64}, "mask": {"size": 2048, "keep_first": 128}}
    dense = {"kind": "dense", "ff": 11008}
    moe = {"kind": "moe", "expert": {"ff": 1408}, "router": {"experts": 64, "top": 6, "groups": {"count": 8, "keep": 4}},
           "shared": {"ff": 2816}}
    return {"architecture": "Gumodra", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6}, "embedding": {"scale": 64.0},
            "layers": [{"type": "attention", "mixer": dict(attn), "mlp": dense}, {"type": "attention", "mixer": dict(attn), "mlp": moe},
                       {"type": "mlstm", "mixer": {"heads": 8, "dim": 256, "vdim": 512, "gate_cap": 15.0}, "mlp": dense},
                       {"type": "attention", "mixer": dict(attn), "mlp": moe}]}


def _sagedra():
    diff = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 256, "scale": 128 ** -0.5, "diff": 0.35, "conv": 4,
            "q_temp": {"coef": 0.1, "every": 1024}}
    pair = {"left": {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 1.0,
                     "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}},
                     "mask": {"size": 2048}},
            "right": {"heads": 32, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}}
    dense = {"kind": "dense", "ff": 11008}
    return {"architecture": "Sagedra", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6}, "embedding": {"scale": 64.0},
            "streams": 4, "logit_softcap": 50.0,
            "layers": [{"type": t, "mixer": dict(m), "mlp": dense} for t, m in 2 * (("attention", diff), ("parallel", pair))]}


def _nelutar():
    left = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 2048}}
    moe = {"kind": "moe", "expert": {"ff": 1408, "limit": 7.0},
           "router": {"experts": 64, "top": 6, "scale": 2.0, "groups": {"count": 8, "keep": 4}}, "shared": {"ff": 2816, "limit": 7.0}}
    pair = {"left": dict(left, rot={"base": 500000.0, "dims": 128}), "right": {"heads": 32, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}}
    both = {"left": dict(left, rot={"base": 10000.0, "dims": 64}, conv=4, softcap=30.0),
            "right": {"heads": 32, "dim": 128, "vdim": 128, "decay": _decays()}, "left_scale": 0.7, "right_scale": 0.4}
    return {"architecture": "Nelutar", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6},
            "embedding": {"bigram": {"buckets": 100003, "mul_prev": 36313, "mul_cur": 27191}},
            "layers": [{"type": "parallel_2", "mixer": both, "mlp": {"kind": "dense", "ff": 11008}},
                       {"type": "parallel", "mixer": pair, "mlp": moe},
                       {"type": "retention", "mixer": {"heads": 32, "dim": 128, "vdim": 128, "decay": _decays(),
                                                       "rot": {"base": 100000.0, "dims": 128}}, "mlp": moe},
                       {"type": "parallel", "mixer": pair, "mlp": moe, "weights_of": 1}]}


def _pemalorn():
    latent = {"heads": 32, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 1536, "kv_rank": 512, "scale": 192 ** -0.5,
              "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}},
              "mask": {"size": 2048}}
    attn = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 500000.0, "dims": 128}}
    moe = {"kind": "moe", "expert": {"ff": 1408}, "router": {"experts": 64, "identity": 16, "top": 6}}
    return {"architecture": "Pemalorn", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6}, "canon": {"taps": 4},
            "token_side": {"dim": 256}, "loop": {"start": 1, "stop": 2, "times": 2},
            "layers": [{"type": "latent_attention", "mixer": dict(latent), "mlp": moe}, {"type": "attention", "mixer": attn, "mlp": moe},
                       {"type": "latent_attention", "mixer": dict(latent), "mlp": moe}]}


def _tirizen():
    gla = {"heads": 32, "dim": 128, "vdim": 128, "tau": 16.0}
    attn = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "q_temp": {"coef": 0.1, "every": 1024}}
    moe = {"kind": "moe", "expert": {"ff": 2112}, "router": {"experts": 64, "top": 6}}
    return {"architecture": "Tirizen", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6}, "embedding": {"scale": 64.0},
            "max_positions": 8192, "residual_mult": 0.1, "streams": 4, "logit_scale": 0.25,
            "layers": [{"type": "gla", "mixer": dict(gla), "mlp": {"kind": "dense", "ff": 16512}},
                       {"type": "attention", "mixer": dict(attn), "mlp": moe}, {"type": "gla", "mixer": dict(gla), "mlp": moe},
                       {"type": "attention", "mixer": dict(attn, kv_from=1), "mlp": moe}]}


SPARSE = {"kernel_size": 32, "kernel_stride": 16, "block_size": 64, "init_blocks": 1, "topk": 64, "window_size": 2048, "dense_len": 8192}
MODELS = {"small": lambda n: _minicpm(n or 24, 1024, 16, 64, 4096, True),
          "8b": lambda n: _minicpm(n or 32, 4096, 32, 128, 16384, False),
          "8b sparse": lambda n: _minicpm(n or 32, 4096, 32, 128, 16384, False, SPARSE),
          "duvulix": lambda n: _duvulix(), "gumodra": lambda n: _gumodra(), "sagedra": lambda n: _sagedra(),
          "nelutar": lambda n: _nelutar(), "pemalorn": lambda n: _pemalorn(), "tirizen": lambda n: _tirizen()}


def model(case):
    """(config.json as a dict, the typed configuration)."""
    raw = MODELS[case["model"]](case["layers"])
    return raw, get_architecture(raw.get("architecture") or raw["architectures"][0]).config_class.from_dict(raw)


def weights(case, seed, config):
    """Random tensors by name.  Where nothing in the configuration says how much a layer adds to the residual, they are
    brought nearer to a trained model's proportions: embeddings of order one, layer scales below one, a mild router (a
    residual that one expert's result outweighs would turn every near tie of the router into another answer)."""
    tensors = random_tensors(config, seed, device=DEVICE)
    if case["model"] in ("nelutar", "pemalorn"):
        for name in tensors:
            if name in ("embed", "bigram"):
                tensors[name] = tensors[name] * 50
            elif name.endswith((".ls1", ".ls2")):
                tensors[name] = tensors[name] * 0.1
            elif case["model"] == "pemalorn" and name.endswith((".router", ".correction")):
                tensors[name] = tensors[name] * 0.4
    return tensors


def token_ids(case, seed):
    """Every sequence's token ids: the prompt's and, behind them, the `new` ones that are fed one by one."""
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, VOCAB, (n + case["new"],), generator=g).tolist() for n in lengths(case)]


# ---------------------------------------------------------------------------------------------------- a pass
def prepare(case, seed):
    raw, config = model(case)
    page = lambda n: -(-n // 64) * 64
    held = [page(n + case["new"]) for n in lengths(case)]
    options = EngineOptions(dtype=case["dtype"], max_tokens=sum(held), max_slots=case["batch"], max_step_tokens=CHUNK, device=DEVICE,
                            max_seq_len=None if case["model"] in ("small", "8b", "8b sparse") else max(held),
                            hip_graph=case["call"] != "prompt",
                            model_options={"sparse": True} if case["model"] == "8b sparse" else {})
    engine = Engine.from_tensors(config, weights(case, seed, config), options)
    ids = token_ids(case, seed)
    state = {"engine": engine, "call": case["call"], "new": case["new"], "ids": ids, "prompts": [t[:n] for t, n in zip(ids, lengths(case))]}
    if case["call"] == "decode":
        slots = [engine.acquire() for _ in ids]
        if any(len(t) > 1 for t in ids):
            engine.step([StepEntry(s, t[:-1]) for s, t in zip(slots, ids) if len(t) > 1])
        state["held"] = [(s, len(t) - 1) for s, t in zip(slots, ids)]
        state["entries"] = [StepEntry(s, t[-1:], [0]) for s, t in zip(slots, ids)]
    return state


def run(state):
    engine = state["engine"]
    if state["call"] == "decode":
        logits = engine.step(state["entries"])
        for slot, length in state["held"]:
            engine.cache.truncate(slot, length)
        return logits
    prompts = state["prompts"]
    slots = [engine.acquire() for _ in prompts]
    out = [engine.step([StepEntry(s, t, [len(t) - 1]) for s, t in zip(slots, prompts)])]
    for i in range(state["new"]):
        out.append(engine.step([StepEntry(s, [t[len(p) + i]], [0]) for s, t, p in zip(slots, state["ids"], prompts)]))
    for s in slots:
        engine.release(s)
    return out


# ---------------------------------------------------------------------------------------------------- work
def _order(raw):
    """Layer indices in the order in which they run."""
    n, loop = len(raw["layers"]), raw.get("loop")
    if not loop:
        return list(range(n))
    a, b = loop["start"], loop["stop"]
    return list(range(a)) + list(range(a, b)) * loop["times"] + list(range(b, n))


def _mixers(raw):
    """(kind, sizes) of every mixer run, pairs taken apart."""
    if "layers" not in raw:
        m = {"heads": raw["num_attention_heads"], "kv_heads": 2, "dim": raw["head_dim"], "vdim": raw["head_dim"]}
        return [("attention", dict(m, sparse=raw.get("sparse_config")))] * raw["num_hidden_layers"]
    out = []
    for i in _order(raw):
        m = raw["layers"][i]["mixer"]
        out += [("attention", m["left"]), ("scan", m["right"])] if "left" in m else [(raw["layers"][i]["type"], m)]
    return out


def _seen(m, p):
    """Keys that the query at position p reads."""
    sparse, mask = m.get("sparse"), m.get("mask")
    if sparse and p + 1 > sparse["dense_len"]:
        return (sparse["topk"] + sparse["window_size"] // sparse["block_size"]) * sparse["block_size"]
    return min(p + 1, mask["size"]) if mask else p + 1


def _pass_work(raw, specs, esize, spans):
    """Bytes and operations of one forward pass over tokens [first, last) of every sequence."""
    n, rows = sum(b - a for a, b in spans), len(spans)
    runs = {}
    for i in (_order(raw) if "layers" in raw else []):
        j = raw["layers"][i].get("weights_of")
        runs[i if j is None else j] = runs.get(i if j is None else j, 0) + 1
    read = flops = 0.0
    tables = 0
    for s in specs:
        numel = math.prod(s.shape)
        at = re.match(r"l(\d+)\.", s.name)
        times = runs.get(int(at.group(1)), 1) if at else raw["loop"]["times"] if s.name == "loop.in" else 1
        if s.init == "table":
            read += n * s.shape[-1] * esize
            tables += 1
        elif re.search(r"\.e\d+\.", s.name):
            r = raw["layers"][int(at.group(1))]["mlp"]["router"]
            share = r["top"] / (r["experts"] + r.get("identity", 0))
            read += numel * esize * (1 - (1 - share) ** n)
            flops += 2 * n * share * numel * times
        elif "lm_head" in s.name or s.name == "head":
            read += numel * esize
            flops += 2 * rows * numel
        else:
            read += numel * esize
            flops += 2 * n * numel * times if len(s.shape) == 2 else 0
    if not any("lm_head" in s.name or s.name == "head" for s in specs):       # the embedding table is the head
        width = raw.get("width") or raw["hidden_size"]
        read += VOCAB * width * esize
        flops += 2 * rows * VOCAB * width
    for kind, m in _mixers(raw):
        H, d, dv = m["heads"], m.get("dim", m.get("state", 0)), m["vdim"]
        for a, b in spans:
            if kind in ("attention", "latent_attention"):
                pairs = sum(_seen(m, p) for p in range(a, b))
                maps = 2 if "diff" in m else 1
                flops += 2 * pairs * H * (maps * (d + m.get("rot_dim", 0)) + maps * dv)
                key = m["kv_rank"] + m["rot_dim"] if kind == "latent_attention" else m["kv_heads"] * (maps * d + dv)
                read += (min(a, _seen(m, b - 1)) + 2 * (b - a)) * key * esize
            else:
                flops += 6 * (b - a) * H * d * dv
                read += 2 * 4 * H * d * dv
    return read + rows * VOCAB * 4, flops


def work(case):
    raw, config = model(case)
    specs = get_architecture(config.architecture).build_model(config).all_weight_specs()
    esize = 4 if case["dtype"] == "float32" else 2
    lens = lengths(case)
    if case["call"] == "decode":
        passes = [[(n - 1, n) for n in lens]]
    else:
        passes = [[(0, n) for n in lens]] + [[(n + i, n + i + 1) for n in lens] for i in range(case["new"])]
    got = [_pass_work(raw, specs, esize, spans) for spans in passes]
    return {"bytes": sum(b for b, _ in got), "flops": sum(f for _, f in got)}


def tolerance(case):
    # Measured by cutting the same prompts into other chunks, so that every product sums in another order: bf16 activations
    # give 0.005 to 0.021 (the deep models most), among it a choice of an expert or a block of keys at a near tie; 32-bit
    # sums are 2.4e-6 from 64 bits.
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.03}


# ---------------------------------------------------------------------------------------------------- in 64 bits
# Whole sequences without a cache, the formulas of the seven models in plain torch, float64.

def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def layer_norm(x, eps):
    return rms(x - x.mean(-1, keepdim=True), eps)


def silu(z):
    return z * torch.sigmoid(z)


def gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


class Weights:
    """The checkpoint's tensors, in float64 when read."""

    def __init__(self, tensors, prefix=""):
        self.tensors, self.prefix = tensors, prefix

    def __contains__(self, name):
        return self.prefix + name in self.tensors

    def __getitem__(self, name):
        return self.tensors[self.prefix + name].double()

    def rows(self, name, ids):
        return self.tensors[self.prefix + name][ids].double()

    def at(self, prefix):
        return Weights(self.tensors, self.prefix + prefix)

    def mul(self, x, name):
        """x W^T, plus the bias that stands beside W, if any."""
        y = x @ self[name].T
        return y + self[name + ".b"] if name + ".b" in self else y


def frequencies(rot):
    """(f_i, magnitude) of a rotation: plain, stretched with a ramp (fast, slow) or by wavelength (low, high)."""
    dims, base = int(rot["dims"]), float(rot["base"])
    i = torch.arange(dims // 2, dtype=torch.float64, device=DEVICE)
    f, sc = base ** (-2.0 * i / dims), rot.get("scaling")
    if not sc:
        return f, 1.0
    factor, original = float(sc["factor"]), float(sc["original"])
    if "low" in sc:
        turns = original * f / (2.0 * math.pi)
        t = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        return (1.0 - t) * f / factor + t * f, 1.0
    at = lambda turns: dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0


def turn(x, f, magnitude=1.0, pairs=False, sign=1.0):
    """x [T, heads, d]: features i and i + len(f) (or neighbours, with `pairs`) rotated by position * f."""
    n = f.numel()
    angle = sign * torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * f
    c, s = (magnitude * torch.cos(angle))[:, None], (magnitude * torch.sin(angle))[:, None]
    a, b = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if pairs else (x[..., :n], x[..., n:2 * n])
    u, v = a * c - b * s, b * c + a * s
    first = torch.stack([u, v], -1).flatten(-2) if pairs else torch.cat([u, v], -1)
    return torch.cat([first, x[..., 2 * n:]], -1)


def rotate(x, rot, pairs=False):
    return turn(x, *frequencies(rot), pairs=pairs) if rot and rot.get("dims") else x


def attend(q, k, v, scale, mask=None, cap=None, sink=None, allowed=None):
    """q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv]: causal softmax attention.  `mask`: a window {size,
    keep_first} or, with {"chunk": n}, chunks; `allowed(a, b)`: [G, b - a, b] for block lists."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    rep, step = H // G, max(32, min(512, (1 << 27) // (H * T)))
    kk, vv, out = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous(), []
    for a in range(0, T, step):
        b = min(T, a + step)
        p, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None]
        see = p >= j
        if mask and "chunk" in mask:
            see &= p // mask["chunk"] == j // mask["chunk"]
        elif mask:
            see &= (p - j < mask["size"]) | (j < mask.get("keep_first", 0))
        see = see[None] if allowed is None else see[None] & allowed(a, b)
        s = (q[a:b].view(b - a, G, rep, -1).permute(1, 2, 0, 3).reshape(G, rep * (b - a), -1) @ kk[:, :, :b]) * scale
        s = cap * torch.tanh(s / cap) if cap else s
        s = s.view(G, rep, b - a, b).masked_fill(~see[:, None], -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(G, rep, 1, 1).expand(G, rep, b - a, 1)], -1)
        w = torch.softmax(s, -1)[..., :b].reshape(G, rep * (b - a), b)
        out.append((w @ vv[:, :b]).view(G, rep, b - a, -1).permute(2, 0, 1, 3).reshape(b - a, H, -1))
    return torch.cat(out)


def scan(q, k, v, keep, beta=None):
    """S <- keep S, then + k v^T (or + k (beta (v - S^T k))^T, the delta rule); o = S^T q.  q, k [T, H, d], v [T, H, dv],
    keep [T, H, 1 or d], beta [T, H]."""
    T, H, d = q.shape
    S, out = q.new_zeros(H, d, v.shape[-1]), torch.empty_like(v)
    keep, kc, qr = keep.expand(T, H, keep.shape[-1])[..., None], k[..., None], q[:, :, None]
    for t in range(T):
        S = S * keep[t]
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - (S * kc[t]).sum(1))
        S = S + kc[t] * u[:, None]
        out[t] = (qr[t] @ S)[:, 0]
    return out


def conv(x, w, bias=None):
    """A causal convolution per channel, the last tap the current token's."""
    taps = w.shape[1]
    pad = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    y = sum(pad[j:j + x.shape[0]] * w[:, j] for j in range(taps))
    return y if bias is None else y + bias


def share(x, heads):
    return x.repeat_interleave(heads // x.shape[1], 1)


def unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


# ---- MiniCPM4
def block_lists(q, k, sc):
    """allowed(a, b) for InfLLM-v2: which of the keys each query and kv head reads (a function of the prefix alone)."""
    T, H, d = q.shape
    G, (ks, st, bs) = k.shape[1], (sc["kernel_size"], sc["kernel_stride"], sc["block_size"])
    n_ck = max((T - ks) // st + 1, 0)
    blocks, local = -(-T // bs), sc["window_size"] // bs
    sums = torch.cat([k.new_zeros(1, G, d), k.cumsum(0)])
    starts = torch.arange(n_ck, device=k.device) * st
    ck = ((sums[starts + ks] - sums[starts]) / ks).permute(1, 2, 0)

    def allowed(a, b):
        p = torch.arange(a, b, device=q.device)
        s = (q[a:b].view(b - a, G, H // G, d).permute(1, 2, 0, 3).reshape(G, -1, d) @ ck).view(G, H // G, b - a, n_ck) * d ** -0.5
        visible = starts[None] + ks <= p[:, None]
        score = torch.nan_to_num(torch.softmax(s.masked_fill(~visible, -math.inf), -1)).sum(1).masked_fill(~visible, -math.inf)
        pool = torch.full((G, b - a, blocks), -math.inf, dtype=q.dtype, device=q.device)
        for half in ((starts // bs), ((starts + ks - 1) // bs)):          # a compressed key overlaps two blocks at most
            pool.scatter_reduce_(2, half.expand(G, b - a, n_ck), score, "amax")
        pool[..., :sc["init_blocks"]] = math.inf
        own = torch.arange(blocks, device=q.device)[None]
        candidate = own <= (p // bs - local)[:, None]
        order = pool.masked_fill(~candidate, -math.inf).sort(dim=-1, descending=True, stable=True).indices
        taken = torch.zeros_like(pool, dtype=torch.bool).scatter_(2, order[..., :min(sc["topk"], blocks)], True) & candidate
        see = taken | ((own > (p // bs - local)[:, None]) & (own <= (p // bs)[:, None]))
        see |= (p + 1 <= sc["dense_len"])[:, None]
        return see.repeat_interleave(bs, -1)[..., :b]
    return allowed


def minicpm(raw, W, ids):
    H, G, d, eps = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"], raw["rms_norm_eps"]
    i = torch.arange(0, d, 2, dtype=torch.float64, device=DEVICE)
    f = 1.0 / (torch.tensor(raw["rope_scaling"]["long_factor"], dtype=torch.float64, device=DEVICE) * raw["rope_theta"] ** (i / d))
    x, branch, T = W.rows("model.embed_tokens.weight", ids) * raw["scale_emb"], raw["scale_depth"] / math.sqrt(raw["num_hidden_layers"]), ids.numel()
    for n in range(raw["num_hidden_layers"]):
        L = W.at(f"model.layers.{n}.")
        a = rms(x, eps) * L["input_layernorm.weight"]
        q, k, v = (L.mul(a, f"self_attn.{t}_proj.weight").view(T, -1, d) for t in "qkv")
        q, k = turn(q, f), turn(k, f)
        allowed = block_lists(q, k, raw["sparse_config"]) if raw.get("sparse_config") and T > raw["sparse_config"]["dense_len"] else None
        x = x + branch * L.mul(attend(q, k, v, d ** -0.5, allowed=allowed).reshape(T, -1), "self_attn.o_proj.weight")
        a = rms(x, eps) * L["post_attention_layernorm.weight"]
        x = x + branch * L.mul(silu(L.mul(a, "mlp.gate_proj.weight")) * L.mul(a, "mlp.up_proj.weight"), "mlp.down_proj.weight")
    return rms(x, eps) * W["model.norm.weight"] * (raw["dim_model_base"] / raw["hidden_size"])


# ---- feed-forwards with routed experts
def experts(h, W, raw_mlp, scores, choice, weights, expert):
    """`choice` [T, n]: the `top` largest are taken (from the best groups, if there are groups); weights(scores taken)."""
    r = raw_mlp["router"]
    groups = r.get("groups")
    if groups:
        per = choice.view(choice.shape[0], groups["count"], -1)
        best = groups["score"](per).topk(groups["keep"], -1).indices
        kept = torch.zeros(per.shape[:2], dtype=torch.bool, device=h.device).scatter_(1, best, True)
        choice = per.masked_fill(~kept[..., None], -math.inf).flatten(1)
    idx = choice.topk(r["top"], -1).indices
    w, out = weights(scores.gather(1, idx)), torch.zeros_like(h)
    for e in range(scores.shape[1]):
        t, j = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            out[t] += w[t, j][:, None] * (expert(h[t], W.at(f"e{e}.")) if e < r["experts"] else h[t])
    return out


def normed(w):
    return w / (w.sum(-1, keepdim=True) + 1e-20)


def grouped(mlp, score):
    return dict(mlp, router=dict(mlp["router"], groups=dict(mlp["router"]["groups"], score=score)))


def silu_ff(h, W):
    return W.mul(silu(W.mul(h, "gate")) * W.mul(h, "up"), "down")


# ---- Duvulix
def duvulix(raw, W, ids):
    eps, x, T, caches = raw["norm"]["eps"], W.rows("embed", ids), ids.numel(), {}
    norm = lambda x, w: rms(x, eps) * (1.0 + w)
    for i, layer in enumerate(raw["layers"]):
        L, m = W.at(f"l{i}."), layer["mixer"]
        M, H, dv, h = L.at("mix."), m["heads"], m["vdim"], norm(x, L["norm1"])
        if layer["type"] == "latent_attention":
            if m.get("kv_from") is None:
                down = M.mul(h, "dkv")
                caches[i] = rms(down[:, :m["kv_rank"]], eps) * M["dkv.norm"], rotate(down[:, None, m["kv_rank"]:], m["rot"])
            c, kr = caches[i if m.get("kv_from") is None else m["kv_from"]]
            q = M.mul(h, "q").view(T, H, -1)
            q = torch.cat([q[..., :m["dim"]], rotate(q[..., m["dim"]:], m["rot"])], -1)
            k = torch.cat([M.mul(c, "uk").view(T, H, -1), kr.expand(T, H, -1)], -1)
            o = attend(q, k, M.mul(c, "uv").view(T, H, dv), m["scale"]) * torch.sigmoid(M.mul(h, "g"))[..., None]
        elif layer["type"] == "attention":
            q, k = (rotate(M.mul(h, t).view(T, -1, m["dim"]), m["rot"]) for t in "qk")
            o = attend(q, k, M.mul(h, "v").view(T, -1, dv), m["scale"], {"chunk": m["mask"]["size"]})
        else:
            N, inner = m["groups"] * m["state"], H * dv
            z, u, dt = M.mul(h, "in").split([inner, inner + 2 * N, H], 1)
            u = silu(conv(u, M["conv"], M["conv.b"]))
            xs, B, C = u[:, :inner].view(T, H, dv), *(share(t.reshape(T, m["groups"], -1), H) for t in u[:, inner:].split(N, 1))
            dt = softplus(dt + M["dt_bias"])
            y = scan(C, dt[..., None] * B, xs, torch.exp(-torch.exp(M["A_log"]) * dt)[..., None]) + M["D"][:, None] * xs
            o = rms((y.reshape(T, inner) * silu(z)).view(T, m["norm_groups"], -1), eps).reshape(T, inner) * M["norm"]
        x = x + norm(M.mul(o.reshape(T, -1), "o"), L["norm1b"])
        z = L.mul(norm(x, L["norm2"]), "mlp.up")
        a, b, c, e = L["mlp.act"].tolist()
        x = x + norm(L.mul(a * rms(z, eps) + b * rms(z ** 2, eps) + c * rms(z ** 3, eps) + e, "mlp.down"), L["norm2b"])
    return norm(x, W["final.norm"])


# ---- Gumodra
def mlstm_scan(q, k, v, a, b):
    T, H, d = q.shape
    S, n, m, out = q.new_zeros(H, d, v.shape[-1]), q.new_zeros(H, d), q.new_zeros(H), torch.empty_like(v)
    for t in range(T):
        new = torch.maximum(b[t] + m, a[t])
        keep, take = torch.exp(b[t] + m - new)[:, None], torch.exp(a[t] - new)[:, None] * k[t]
        S, n, m = keep[..., None] * S + take[..., None] * v[t][:, None], keep * n + take, new
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
        out[t] = (q[t][:, None] @ S)[:, 0] / den[:, None]
    return out


def gumodra(raw, W, ids):
    eps, T = raw["norm"]["eps"], ids.numel()
    x = W.rows("embed", ids) * raw["embedding"]["scale"]
    for i, layer in enumerate(raw["layers"]):
        L, m = W.at(f"l{i}."), layer["mixer"]
        M, h, F = L.at("mix."), rms(x, eps) * L["norm1"], L.at("mlp.")
        if layer["type"] == "attention":
            q, v = M.mul(h, "q").view(T, -1, m["dim"]), M.mul(h, "k").view(T, -1, m["dim"])
            q, k = rotate(rms(q, eps) * M["q.norm"], m["rot"]), rotate(rms(v, eps) * M["k.norm"], m["rot"])
            o = attend(q, k, v, m["scale"], m["mask"], sink=M["sink"] if "sink" in M else None).reshape(T, -1)
        else:
            q, k = M.mul(h, "q").view(T, -1, m["dim"]) * m["dim"] ** -0.5, M.mul(h, "k").view(T, -1, m["dim"])
            capped = lambda t: m["gate_cap"] * torch.tanh(M.mul(h, t) / m["gate_cap"])
            o = mlstm_scan(q, k, M.mul(h, "v").view(T, -1, m["vdim"]), capped("i"), torch.nn.functional.logsigmoid(capped("f")))
            o = rms(o, eps).reshape(T, -1) * M["norm"] * torch.sigmoid(M.mul(h, "g"))
        y = torch.sigmoid(L.mul(h, "rg1")) * M.mul(o, "o")
        if layer["mlp"]["kind"] == "dense":
            f = silu_ff(h, F)
        else:
            s = torch.softmax(F.mul(h, "router"), -1)
            f = experts(h, F, grouped(layer["mlp"], lambda g: g.max(-1).values), s, s + F["correction"], normed, silu_ff)
            f = f + torch.sigmoid(F.mul(h, "shared.sg")) * silu_ff(h, F.at("shared."))
        x = x + y + torch.sigmoid(L.mul(h, "rg2")) * f
    return rms(x, eps) * W["final.norm"]


# ---- Sagedra and Nelutar
def delta(h, W, m, eps, channels):
    """The gated delta rule, one decay a head or (with `channels`) one a head and key channel."""
    T, H, G, d, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (silu(conv(W.mul(h, t), W[t + ".conv"])) for t in "qkv")
    q, k = unit(q.view(T, G, d)) * d ** -0.5, unit(k.view(T, G, d))
    a = (W.mul(W.mul(h, "a1"), "a2") if channels else W.mul(h, "a")) + W["dt_bias"]
    keep = torch.exp(-torch.exp(W["A_log"])[:, None] * softplus(a).view(T, H, -1))
    o = rms(scan(share(q, H), share(k, H), v.view(T, H, dv), keep, torch.sigmoid(W.mul(h, "b"))), eps) * W["norm"]
    gate = torch.sigmoid(W.mul(W.mul(h, "g1"), "g2")) if channels else silu(W.mul(h, "g"))
    return W.mul(o.reshape(T, -1) * gate, "o")


def mean_of_normed(a, b, W, eps):
    return 0.5 * (rms(a, eps) * W["left.out"] + rms(b, eps) * W["right.out"])


def sagedra(raw, W, ids):
    eps, T = raw["norm"]["eps"], ids.numel()
    X = (W.rows("embed", ids) * raw["embedding"]["scale"]).expand(raw["streams"], -1, -1)

    def pair(h, M, m):
        a, A = m["left"], M.at("left.")
        q, k = (rms(rotate(A.mul(h, t).view(T, -1, a["dim"]), a["rot"]), eps) for t in "qk")
        o = attend(q, k, A.mul(h, "v").view(T, -1, a["vdim"]), a["scale"], a["mask"]).reshape(T, -1)
        return mean_of_normed(A.mul(o * torch.sigmoid(A.mul(h, "g")), "o"), delta(h, M.at("right."), m["right"], eps, False), M, eps)

    def differential(h, M, m):
        q, k, v = (conv(M.mul(h, t), M[t + ".conv"]) for t in "qkv")
        p = torch.arange(T, dtype=torch.float64, device=h.device)
        warm = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((p + 1) / m["q_temp"]["every"]) + 1.0)
        q, k, v = q.view(T, -1, 2, m["dim"]) * warm[:, None, None, None], k.view(T, -1, 2, m["dim"]), v.view(T, -1, m["vdim"])
        one, two = (attend(q[:, :, j], k[:, :, j], v, m["scale"]) for j in (0, 1))
        lam = torch.exp((M["lq1"] * M["lk1"]).sum()) - torch.exp((M["lq2"] * M["lk2"]).sum()) + m["diff"]
        return M.mul((rms(one - lam * two, eps) * (1.0 - m["diff"])).reshape(T, -1), "o")

    def sub(X, L, n, fn):
        h = layer_norm(torch.einsum("s,std->td", L[f"hc{n}.in"], X), eps) * L[f"norm{n}"]
        return torch.einsum("st,snd->tnd", L[f"hc{n}.mix"], X) + L[f"hc{n}.out"][:, None, None] * fn(h)[None]

    for i, layer in enumerate(raw["layers"]):
        L, mixer = W.at(f"l{i}."), differential if layer["type"] == "attention" else pair
        X = sub(X, L, 1, lambda h: mixer(h, L.at("mix."), layer["mixer"]))
        X = sub(X, L, 2, lambda h: L.mul(gelu(L.mul(h, "mlp.gate")) * L.mul(h, "mlp.up"), "mlp.down"))
    return layer_norm(X.sum(0), eps) * W["final.norm"]


def nelutar(raw, W, ids):
    eps, T, big = raw["norm"]["eps"], ids.numel(), raw["embedding"]["bigram"]
    rows = torch.full_like(ids, big["buckets"])
    rows[1:] = (ids[:-1] * big["mul_prev"] + ids[1:] * big["mul_cur"]) % big["buckets"]
    x = W.rows("embed", ids) + W.rows("bigram", rows)

    def left(h, A, a, normal):
        q, k, v = (conv(A.mul(h, t), A[t + ".conv"]) if a.get("conv") else A.mul(h, t) for t in "qkv")
        q, k = (rotate(t.view(T, -1, a["dim"]), a["rot"], pairs=True) for t in (q, k))
        q, k = (rms(q, eps), rms(k, eps)) if normal else (q, k)
        return A.mul(attend(q, k, v.view(T, -1, a["vdim"]), a["scale"], a["mask"], a.get("softcap")).reshape(T, -1), "o")

    def decaying(q, k, v, m):
        keep = torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE)[None, :, None].expand(T, -1, -1)
        return scan(q, k, v, keep)

    def mixer(h, M, kind, m):
        if kind == "retention":
            q, k = (rotate(M.mul(h, t).view(T, -1, m["dim"]), m["rot"]) for t in "qk")
            o = rms(decaying(q, k * m["dim"] ** -0.5, M.mul(h, "v").view(T, -1, m["vdim"]), m), eps)
            return M.mul(o.reshape(T, -1) * silu(M.mul(h, "g")), "o")
        if kind == "parallel":
            return mean_of_normed(left(h, M.at("left."), m["left"], False), delta(h, M.at("right."), m["right"], eps, True), M, eps)
        R, r = M.at("right."), m["right"]
        o = decaying(*(silu(R.mul(h, t)).view(T, r["heads"], -1) for t in "qkv"), r).reshape(T, -1)
        o = R.mul(rms(o, eps) * R["norm"] * torch.sigmoid(R.mul(h, "g")), "o")
        return m["left_scale"] * left(h, M.at("left."), m["left"], True) + m["right_scale"] * o

    def clamped(limit):
        def expert(h, E):
            g, u = torch.clamp(E.mul(h, "gate"), max=limit), torch.clamp(E.mul(h, "up"), -limit, limit)
            return E.mul(g * torch.sigmoid(1.702 * g) * (u + 1.0), "down")
        return expert

    for i, layer in enumerate(raw["layers"]):
        L, mlp = W.at(f"l{layer.get('weights_of', i)}."), layer["mlp"]
        h, F = rms(x, eps) * L["norm1"], L.at("mlp.")
        if mlp["kind"] == "dense":
            f = silu_ff(h, F)
        else:
            s, scale = torch.sigmoid(F.mul(h, "router")), mlp["router"]["scale"]
            choice = s + F["correction"] if "correction" in F else s
            f = experts(h, F, grouped(mlp, lambda g: g.topk(2, -1).values.sum(-1)), s, choice, lambda w: normed(w) * scale,
                        clamped(mlp["expert"]["limit"])) + clamped(mlp["shared"]["limit"])(h, F.at("shared."))
        x = x + L["ls1"] * mixer(h, L.at("mix."), layer["type"], layer["mixer"]) + L["ls2"] * f
    return rms(x, eps) * W["final.norm"]


# ---- Pemalorn
def pemalorn(raw, W, ids):
    eps, T, side = raw["norm"]["eps"], ids.numel(), raw["token_side"]["dim"]
    x = first = W.rows("embed", ids)
    done = 0
    for i in _order(raw):
        layer, L, m = raw["layers"][i], W.at(f"l{i}."), raw["layers"][i]["mixer"]
        if i == raw["loop"]["start"]:
            x, done = W.mul(torch.cat([x, first], -1), "loop.in") + W["loop.step"][done], done + 1
        h = layer_norm(x, eps) * L["norm1"]
        M, F = L.at("mix."), L.at("mlp.")
        h1, h2 = (h + conv(h, L[f"canon{n}"]) for n in (1, 2))
        if layer["type"] == "attention":
            back = float(m["rot"]["base"]) ** (-2.0 * torch.arange(m["vdim"] // 2, dtype=torch.float64, device=DEVICE) / m["vdim"])
            q, k = (rotate(M.mul(h1, t).view(T, -1, m["dim"]), m["rot"]) for t in "qk")
            v = turn(M.mul(h1, "v").view(T, -1, m["vdim"]), back)
            o = turn(attend(q * M["temp"][:, None], k, v, m["scale"], sink=M["sink"]), back, sign=-1.0)
            o = o * torch.sigmoid(M.mul(h1, "g"))[..., None]
        else:
            H, R, d = m["heads"], m["kv_rank"], m["dim"]
            q = M.mul(rms(M.mul(h1, "dq"), eps) * M["dq.norm"], "uq").view(T, H, -1)
            down = M.mul(h1, "dkv")
            c, kr = rms(down[:, :R], eps) * M["dkv.norm"], rotate(down[:, None, R:], m["rot"], pairs=True)
            q = torch.cat([q[..., :d], rotate(q[..., d:], m["rot"], pairs=True)], -1)
            k = torch.cat([M.mul(c, "uk").view(T, H, d), kr.expand(T, H, -1)], -1)
            o = attend(q, k, M.mul(c, "uv").view(T, H, -1), m["scale"], m["mask"], sink=M["sink"])
            o = o.reshape(T, -1) * torch.sigmoid(M.mul(h1, "g"))
        s = torch.softmax(F.mul(h2, "router"), -1)
        x = x + M.mul(o.reshape(T, -1), "o") + experts(h2, F, layer["mlp"], s, s + F["correction"], lambda w: w, silu_ff)
        e = W.rows("side.embed", ids)[:, i * side:(i + 1) * side]
        x = x + rms(L.mul(gelu(L.mul(x, "side.gate")) * e, "side.proj"), eps) * L["side.norm"]
    return layer_norm(x, eps) * W["final.norm"]


# ---- Tirizen
def tirizen(raw, W, ids):
    eps, T, kept = raw["norm"]["eps"], ids.numel(), {}
    x = W.rows("embed", ids) * raw["embedding"]["scale"] + W.rows("pos", torch.arange(T, device=ids.device))
    X = x.expand(raw["streams"], -1, -1)

    def gla(h, M, m, i):
        q, k, v = (M.mul(h, t).view(T, m["heads"], -1) for t in "qkv")
        keep = torch.exp(torch.nn.functional.logsigmoid(M.mul(M.mul(h, "a1"), "a2")) / m["tau"]).view(T, m["heads"], -1)
        o = rms(scan(q * m["dim"] ** -0.5, k, v, keep), eps) * M["norm"]
        return M.mul(o.reshape(T, -1) * silu(M.mul(h, "g")), "o")

    def attention(h, M, m, i):
        p = torch.arange(T, dtype=torch.float64, device=h.device)
        warm = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((p + 1) / m["q_temp"]["every"]) + 1.0)
        q = (rms(M.mul(h, "q"), eps) * M["q.norm"] * warm[:, None]).view(T, m["heads"], -1)
        if m.get("kv_from") is None:
            kept[i] = (rms(M.mul(h, "k"), eps) * M["k.norm"]).view(T, -1, m["dim"]), M.mul(h, "v").view(T, -1, m["vdim"])
        o = attend(q, *kept[i if m.get("kv_from") is None else m["kv_from"]], m["scale"])
        return M.mul((o * torch.sigmoid(M.mul(h, "g"))[..., None]).reshape(T, -1), "o")

    def plain(h, E):
        return E.mul(torch.clamp(E.mul(h, "up"), min=0.0) ** 2, "down")

    def feed(h, F, mlp):
        if mlp["kind"] == "dense":
            return plain(h, F)
        z = F.mul(h, "router")
        return experts(h, F, mlp, z, z, lambda w: torch.softmax(w, -1), plain)

    def sub(X, L, n, fn):
        h = rms(torch.einsum("s,std->td", L[f"hc{n}.in"], X), eps) * L[f"norm{n}"]
        return torch.einsum("st,snd->tnd", L[f"hc{n}.mix"], X) + raw["residual_mult"] * L[f"hc{n}.out"][:, None, None] * fn(h)[None]

    for i, layer in enumerate(raw["layers"]):
        L, mixer = W.at(f"l{i}."), gla if layer["type"] == "gla" else attention
        X = sub(X, L, 1, lambda h: mixer(h, L.at("mix."), layer["mixer"], i))
        X = sub(X, L, 2, lambda h: feed(h, L.at("mlp."), layer["mlp"]))
    return rms(X.sum(0), eps) * W["final.norm"] * raw["logit_scale"]


PLAIN = {"small": minicpm, "8b": minicpm, "8b sparse": minicpm, "duvulix": duvulix, "gumodra": gumodra, "sagedra": sagedra,
         "nelutar": nelutar, "pemalorn": pemalorn, "tirizen": tirizen}


def exact(case, seed):
    raw, config = model(case)
    # the longest ones would take over 20 seconds: all layers of the 8b model over many whole contexts
    if sum(lengths(case)) * (raw.get("num_hidden_layers") or 0) * (raw.get("hidden_size") or 0) ** 2 > 2.4e13:
        return None
    W = Weights(weights(case, seed, config))
    head = next((t for t in ("lm_head.weight", "head") if t in W), None) or next(t for t in ("model.embed_tokens.weight", "embed") if t in W)
    last = []
    for ids in token_ids(case, seed):
        h = PLAIN[case["model"]](raw, W, torch.tensor(ids, device=DEVICE))
        last.append(h[len(ids) - 1 - case["new"]:])
    H = W[head].T.contiguous()
    out = [torch.stack([h[i] for h in last]) @ H for i in range(case["new"] + 1)]
    if raw.get("logit_softcap"):
        out = [raw["logit_softcap"] * torch.tanh(t / raw["logit_softcap"]) for t in out]
    return out[0] if case["call"] == "decode" else out
