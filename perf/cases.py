"""The work that programs give this engine, as cases to be timed and compared.

A case is what a serving or scoring program does with one engine: requests are admitted, their
prompts are read (whole, several a step, or in portions beside requests that already decode), further
tokens follow one a step, and the pages and slots go back.  The tokens after the prompts are given,
as in a trace replay: two correct implementations then compute the same logits up to their rounding,
where one flipped choice of a token would make everything after it incomparable.  The choice of a
token is a case of its own.

Models are the configurations of ``yalis_amd.models.presets`` with random weights.  The designs whose
experts are chosen by a router's scores (Mesolix, Bekedra, Zimupel) are not among the cases: which
expert wins a near tie is decided by rounding, so no tolerance tells a right implementation from a
wrong one; their mixers share the kernels of those that are here (attention, latent attention,
state scans, grouped experts chosen by Suranex's table).

The two larger Llama shapes run at full width with fewer layers (``LAYERS``; ``bench.py --layers`` does
the same): layers are alike, and through all 32 of them two right bfloat16 implementations differ by
3.3 % in the logits (measured: the same tokens read whole, 48 and 17 at a time), which says nothing any
more; through 12 of them by 1.9 %.

The engine (weights, pool, captured graphs) is made once per model and type and kept, as a program
keeps it; a seed makes other prompts.
"""
import hashlib
import math

import numpy as np
import torch

from yalis_amd import InferenceConfig, LLMEngine, SamplingParams
from yalis_amd.config.runtime import EngineConfig
from yalis_amd.engine.factory import tensor_specs_for
from yalis_amd.engine.step import StepEntry
from yalis_amd.models.presets import SHAPES

F = torch.float64
WEIGHT_SEED = 0
MAX_SEQS = 65        # requests alive at once: 64 that decode and one whose prompt is being read
MAX_LEN = 4096       # longest sequence
STEP_TOKENS = 8192   # most tokens of one step
POOL_PAGES = 1024    # of 64 tokens
LAYERS = {"8b": 12, "3b": 14}


def _config(case):
    config = dict(SHAPES[case["model"]][1])
    if case["model"] in LAYERS:
        config["num_hidden_layers"] = LAYERS[case["model"]]
    return config


# ------------------------------------------------------------------------------------- the cases
def _case(name, kind, model, dtype="bfloat16", prompts=1, shortest=0, longest=0, steps=0, long=0, portion=0):
    return {"name": name, "kind": kind, "model": model, "dtype": dtype, "prompts": prompts, "shortest": shortest, "longest": longest,
            "steps": steps, "long": long, "portion": portion}


def listed():
    return [
        # a chat with the smallest of the Llama shapes: a short prompt, an answer, one request (latency of a step)
        _case("chat_1b", "generate", "1b", shortest=37, longest=37, steps=16),
        # the headline workload: eight 1,024-token prompts and 32 tokens each
        _case("generate_8b_8", "generate", "8b", prompts=8, shortest=1024, longest=1024, steps=32),
        # a full batch of short questions of different lengths
        _case("generate_8b_64", "generate", "8b", prompts=64, shortest=65, longest=191, steps=8),
        # reading one document: time to the first token
        _case("prefill_8b_2048", "generate", "8b", shortest=2048, longest=2048),
        # continuous batching: a long prompt arrives in portions beside 32 requests that decode
        _case("mixed_3b", "mixed", "3b", prompts=32, shortest=90, longest=160, long=1920, portion=480),
        # scoring a text: the logits of every position
        _case("score_1b", "score", "1b", shortest=999, longest=999),
        # the 32-bit engine, as a reference run or a model that needs it
        _case("float32_1b", "generate", "1b", dtype="float32", prompts=2, shortest=200, longest=311, steps=4),
        # windowed attention, gated linear recurrence, experts chosen by a table: ragged prompts and answers
        _case("suranex_2k", "generate", "suranex-2k", prompts=4, shortest=500, longest=901, steps=16),
        # latent attention, delta rule, gated linear attention: reading one document
        _case("prefill_nutavik_2k", "generate", "nutavik-2k", shortest=2048, longest=2048),
        # the same design, wider: a batch of short questions and answers
        _case("generate_nutavik_4k", "generate", "nutavik-4k", prompts=8, shortest=70, longest=130, steps=24),
        # delta rule with a decay per channel, chunked attention beside time mixing: ragged prompts and answers
        _case("rafusun_2k", "generate", "rafusun-2k", prompts=8, shortest=111, longest=700, steps=16),
        # choosing a batch's tokens: top-k, temperature and top-p over the Llama 3 vocabulary
        _case("sample_8", "sample", "8b", prompts=8),
    ]


# the range of every kind and model: (model, dtype, kinds, most prompts, longest prompt, most tokens read in all, most steps)
_RANGES = [
    ("1b", "bfloat16", ("generate", "score"), 64, 2048, 8192, 24),
    ("3b", "bfloat16", ("generate", "mixed"), 64, 2048, 8192, 16),
    ("8b", "bfloat16", ("generate", "generate"), 64, 2048, 8192, 16),
    ("1b", "float32", ("generate",), 4, 300, 600, 4),
    ("suranex-2k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("suranex-4k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("nutavik-2k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("nutavik-4k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("rafusun-2k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("rafusun-4k", "bfloat16", ("generate",), 16, 2048, 4096, 16),
    ("8b", "bfloat16", ("sample",), 64, 1, 64, 0),
]


def _log_uniform(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))))


def draw(rng):
    model, dtype, kinds, most, longest, total, most_steps = rng.choice(_RANGES)
    kind = rng.choice(kinds)
    if kind == "sample":
        return _unnamed("sample", model, dtype, prompts=_log_uniform(rng, 1, most))
    if kind == "score":
        n = _log_uniform(rng, 17, 1500)
        return _unnamed("score", model, dtype, shortest=n, longest=n)
    if kind == "mixed":
        portion = rng.choice((224, 480, 992)) + rng.choice((0, 0, rng.randrange(32)))
        lo = _log_uniform(rng, 16, 200)
        return _unnamed("mixed", model, dtype, prompts=_log_uniform(rng, 2, 32), shortest=lo, longest=lo + rng.randrange(100),
                        long=portion * rng.randint(1, 1950 // portion) + rng.randrange(portion), portion=portion)
    n = _log_uniform(rng, 1, most)
    hi = _log_uniform(rng, 16, min(longest, max(16, total // n)))
    lo = hi if n == 1 else max(1, int(hi * rng.uniform(0.3, 1.0)))
    return _unnamed("generate", model, dtype, prompts=n, shortest=lo, longest=hi, steps=rng.randint(0, most_steps))


def _unnamed(kind, model, dtype, **sizes):
    case = _case("", kind, model, dtype, **sizes)
    del case["name"]
    return case


# ------------------------------------------------------------------------------- what a case runs
def _lengths(case):
    n, lo, hi = case["prompts"], case["shortest"], case["longest"]
    return [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)]


def _script(case):
    """The steps of a case: lists of (request, first token, tokens, wanted places)."""
    lengths = _lengths(case)
    done = [0] * len(lengths)
    steps, step, room = [], [], STEP_TOKENS
    for r, length in enumerate(lengths):  # prompts packed into steps, one that does not fit is cut
        while done[r] < length:
            n = min(room, length - done[r])
            last = done[r] + n == length
            want = list(range(n)) if case["kind"] == "score" else [n - 1] if last else []
            step.append((r, done[r], n, want))
            done[r] += n
            room -= n
            if room == 0:
                steps.append(step)
                step, room = [], STEP_TOKENS
    if step:
        steps.append(step)
    if case["kind"] == "mixed":
        at, new = 0, len(lengths)
        while at < case["long"]:
            n = min(case["portion"], case["long"] - at)
            step = [(r, done[r], 1, [0]) for r in range(len(lengths))]
            step.append((new, at, n, [n - 1] if at + n == case["long"] else []))
            done = [d + 1 for d in done]
            at += n
            steps.append(step)
        done.append(at)
    for _ in range(case["steps"]):
        steps.append([(r, done[r], 1, [0]) for r in range(len(lengths))])
        done = [d + 1 for d in done]
    return steps, done


def _sequences(case, seed):
    """Every request's tokens, from the seed."""
    rng = np.random.RandomState(seed % (1 << 32))
    config = _config(case)
    vocab = config.get("vocab", config.get("vocab_size"))
    return [rng.randint(0, vocab, n).tolist() for n in _script(case)[1]]


_engine = None  # (model, dtype), LLMEngine: the one that is kept


def _engine_for(case):
    global _engine
    key = (case["model"], case["dtype"])
    if _engine is None or _engine[0] != key:
        _engine = None
        torch.cuda.empty_cache()
        config = EngineConfig(page_size=64, num_pages=POOL_PAGES, max_num_seqs=MAX_SEQS, max_model_len=MAX_LEN,
                              max_num_batched_tokens=STEP_TOKENS, dtype=case["dtype"])
        limits = InferenceConfig(max_batch_size=MAX_SEQS, max_length_of_generated_sequences=MAX_LEN, temperature=0.0)
        precision = {"bfloat16": "bf16", "float32": "fp32"}[case["dtype"]]
        _engine = key, LLMEngine.from_random(_config(case), limits, precision=precision, seed=WEIGHT_SEED, engine_config=config)
    return _engine[1]


class _Sampling:
    """A sampler, a batch's logits and its requests' parameters."""

    def __init__(self, case, seed):
        from yalis_amd.ops.hip import HipOps
        from yalis_amd.sampling.sampler import Sampler

        vocab, rows = SHAPES[case["model"]][1]["vocab_size"], case["prompts"]
        g = torch.Generator(device="cuda").manual_seed(seed)
        # a few dozen likely tokens above a wide tail, as a trained model gives
        self.logits = torch.randn(rows, vocab, device="cuda", generator=g) * 2.5
        likely = torch.randint(0, vocab, (rows, 50), device="cuda", generator=g)
        self.logits.scatter_add_(1, likely, torch.full((rows, 50), 9.0, device="cuda"))
        self.params = [SamplingParams(temperature=0.7, top_k=50, top_p=0.8, seed=(seed * 1000003 + i) & 0x7FFFFFFF) for i in range(rows)]
        self.sampler = Sampler(HipOps("cuda:0"), "cuda:0")
        self.prepared = self.sampler.prepare(self.params, [0] * rows)


class _Requests:
    """An engine and the requests that it is about to serve."""

    def __init__(self, case, seed):
        self.runner = _engine_for(case).runner
        sequences = _sequences(case, seed)
        self.steps = [[StepEntry(r, sequences[r][a: a + n], want) for r, a, n, want in step] for step in _script(case)[0]]


def prepare(case, seed):
    return _Sampling(case, seed) if case["kind"] == "sample" else _Requests(case, seed)


def run(state):
    if isinstance(state, _Sampling):
        return state.sampler.sample_prepared(state.logits, state.prepared, 0)
    runner, out = state.runner, []
    for step in state.steps:
        for e in step:
            if not runner.is_live(e.request) and not runner.admit(e.request):
                raise RuntimeError("no slot left")
            if not runner.reserve(e.request, len(e.tokens)):
                raise RuntimeError("no pages left")
        logits = runner.step(step)
        if logits.shape[0]:
            # a step of single tokens leaves its logits in a buffer that the next such step writes again
            out.append(logits.clone() if all(len(e.tokens) == 1 for e in step) else logits)
    for request in list(runner.cached):
        runner.release(request)
    return out


# ----------------------------------------------------------------------- what it cannot do without
def _experts(config):
    for layer in config.get("layers", ()):
        if layer.get("mlp") and layer["mlp"].get("kind") == "moe":
            yield layer["mlp"]


def work(case):
    config = _config(case)
    if case["kind"] == "sample":
        # the logits read once, a token a row written
        return {"bytes": 4.0 * case["prompts"] * config["vocab_size"] + 4.0 * case["prompts"], "flops": 0.0}
    size = 2 if case["dtype"] == "bfloat16" else 4
    specs = tensor_specs_for(dict(config))
    vocab = config.get("vocab", config.get("vocab_size"))
    width = config.get("width", config.get("hidden_size"))
    dense = sum(math.prod(s.shape) for n, s in specs.items()
                if s.kind == "float" and len(s.shape) > 1 and s.shape[0] != vocab and "bigram" not in n and ".mlp.e" not in n)
    expert, top, experts = 0, 0, 0
    for f in _experts(config):
        expert, top, experts = 3 * width * f["expert"]["ff"], f["router"]["top"], f["router"]["experts"]
    n_moe = len(list(_experts(config)))
    # per layer: (numbers cached for a position, key reads and value reads of a position and head, heads, window) and
    # (numbers of a request's matrix states)
    attention, states = [], []
    if "layers" not in config:
        g, d = config["num_key_value_heads"], config["head_dim"]
        attention = [(2 * g * d, 2 * d, config["num_attention_heads"], None)] * config["num_hidden_layers"]
    for layer in config.get("layers", ()):
        m = layer["mixer"]
        if layer["type"] == "latent_attention":
            attention.append((m["kv_rank"] + m["rot_dim"], m["dim"] + m["rot_dim"] + m["vdim"], m["heads"], None))
        elif layer["type"] in ("attention", "parallel"):
            a = m.get("left", m)
            attention.append((a["kv_heads"] * (a["dim"] + a["vdim"]), a["dim"] + a["vdim"], a["heads"], a["mask"]["size"]))
        if layer["type"] == "parallel":
            states.append(m["right"]["heads"] * m["right"]["dim"] ** 2)
        elif layer["type"] in ("delta", "gla", "channel_delta"):
            states.append(m["heads"] * m["dim"] * m["vdim"])
    moved = flops = 0.0
    for step in _script(case)[0]:
        tokens = sum(n for _, _, n, _ in step)
        rows = sum(len(want) for *_, want in step)
        moved += size * (dense + n_moe * expert * min(experts, tokens * top) + tokens * width) + (size * vocab * width + 4.0 * rows * vocab if rows else 0)
        flops += 2.0 * tokens * (dense + n_moe * expert * top) + 2.0 * rows * vocab * width
        for _, first, n, _ in step:
            for cached, per_key, heads, window in attention:
                reach = min(window or first + n, first + n)
                moved += size * cached * (min(first, reach) + n)
                seen = n * first + n * (n + 1) / 2 if not window else n * min(window, first + n / 2)
                flops += 2.0 * heads * per_key * seen
            for numbers in states:
                moved += 4.0 * numbers * (1 + (first > 0))
                flops += 6.0 * numbers * n
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"  # the choice is a function of the logits and the request's own stream of numbers
    if case["dtype"] == "float32":
        return {"rel": 2e-5}  # 5e-6 from the 64-bit logits
    # what two right implementations differ by (the same tokens read whole, 48 and 17 at a time): 1.1 % for the shallow
    # designs, 1.6 to 2 % for the deeper ones; a sum in another order flips bfloat16 roundings, and every layer passes them on
    return {"rel": 0.03}


# ------------------------------------------------------------------------- the same in 64 bits
def _weights(config, dtype):
    """name -> the tensor that the engine's random weights hold under it, in 64 bits."""
    specs = tensor_specs_for(dict(config))
    device = "cuda:0" if torch.cuda.is_available() else "cpu"

    def get(name):
        spec = specs[name]
        digest = hashlib.sha256(f"{WEIGHT_SEED}:{name}".encode()).digest()
        g = torch.Generator(device=device).manual_seed(int.from_bytes(digest[:8], "little") & 0x7FFFFFFFFFFFFFFF)
        if spec.kind == "int":  # every row: different numbers, in random order
            draws = torch.rand((*spec.shape[:-1], spec.init[1]), generator=g, device=device)
            return draws.argsort(dim=-1)[..., : spec.shape[-1]]
        t = torch.randn(spec.shape, generator=g, device=device, dtype=torch.float32) * spec.init[1]
        return ((1.0 + t if spec.init[0] == "one_plus_normal" else t).to(getattr(torch, dtype))).to(F)

    return get


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _turn(x, angle, pairs, mag=1.0):
    """x [n, ..., d], angle [n, r / 2]: the first r elements of every vector turn, in pairs (i, i + r/2) or (2i, 2i + 1)."""
    r = 2 * angle.shape[-1]
    shape = [x.shape[0]] + [1] * (x.dim() - 2) + [r // 2]
    c, s = (torch.cos(angle) * mag).view(shape), (torch.sin(angle) * mag).view(shape)
    a, b = (x[..., : r // 2], x[..., r // 2: r]) if pairs == "half" else (x[..., 0:r:2], x[..., 1:r:2])
    u, v = a * c - b * s, b * c + a * s
    turned = torch.cat([u, v], -1) if pairs == "half" else torch.stack([u, v], -1).flatten(-2)
    return torch.cat([turned, x[..., r:]], -1)


def _frequencies(dims, base, yarn, device):
    """Angle per position of every pair, and what a stretched rotation multiplies with."""
    i = torch.arange(dims // 2, dtype=F, device=device)
    f = base ** (-2.0 * i / dims)
    if not yarn:
        return f, 1.0
    where = lambda turns: dims * math.log(yarn["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(where(yarn["fast"])), 0), min(math.ceil(where(yarn["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / yarn["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(yarn["factor"]) + 1.0


def _attend(q, k, v, scale, cap=None, mask=None, sink=False):
    """q [n, H, d], k and v [n, G, .]: softmax attention over the keys that ``mask`` [n, n] shows (by default all earlier ones)."""
    n, share = q.shape[0], q.shape[1] // k.shape[1]
    if mask is None:
        mask = torch.ones(n, n, dtype=torch.bool, device=q.device).tril()
    out = torch.empty(n, q.shape[1], v.shape[-1], dtype=F, device=q.device)
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // share].T * scale
        s = (cap * torch.tanh(s / cap) if cap else s).masked_fill(~mask, -math.inf)
        if sink:  # a key of score 0 without a value
            s = torch.cat([s, torch.zeros(n, 1, dtype=F, device=q.device)], 1)
        out[:, h] = torch.softmax(s, -1)[:, :n] @ v[:, h // share]
    return out


def _convolution(x, taps):
    """Per channel over time, zeros before the start, the last tap on the current token."""
    n, t = x.shape[0], taps.shape[1]
    padded = torch.cat([torch.zeros(t - 1, x.shape[1], dtype=F, device=x.device), x])
    return sum(padded[j: j + n] * taps[:, j] for j in range(t))


def _positions(n, f):
    return torch.arange(n, dtype=F, device=f.device)[:, None] * f


class _Llama:
    def __init__(self, config, get):
        self.c, self.layers, self.embed = config, config["num_hidden_layers"], get("model.embed_tokens.weight")
        self.final = get("model.norm.weight")
        self.head = self.embed if config["tie_word_embeddings"] else get("lm_head.weight")
        d = config["head_dim"]
        f = config["rope_theta"] ** (-torch.arange(0, d, 2, dtype=F, device=self.embed.device) / d)
        if config["rope_scaling"]:
            r = config["rope_scaling"]
            ratio = r["original_max_position_embeddings"] * f / (2 * math.pi)
            smooth = ((ratio - r["low_freq_factor"]) / (r["high_freq_factor"] - r["low_freq_factor"])).clamp(0.0, 1.0)
            f = (1 - smooth) * f / r["factor"] + smooth * f
        self.f = f

    def start(self, tokens):
        return self.embed[tokens]

    def names(self, i):
        p = f"model.layers.{i}."
        parts = ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj",
                 "input_layernorm", "post_attention_layernorm")
        return {s.split(".")[-1]: p + s + ".weight" for s in parts}

    def layer(self, i, W, x, tokens, memo):
        c, eps, n = self.c, self.c["rms_norm_eps"], x.shape[0]
        h = _unit(x, eps) * W["input_layernorm"]
        q, k, v = ((h @ W[s + "_proj"].T).view(n, -1, c["head_dim"]) for s in "qkv")
        angle = _positions(n, self.f)
        o = _attend(_turn(q, angle, "half"), _turn(k, angle, "half"), v, c["head_dim"] ** -0.5)
        x = x + o.reshape(n, -1) @ W["o_proj"].T
        h = _unit(x, eps) * W["post_attention_layernorm"]
        return x + (_silu(h @ W["gate_proj"].T) * (h @ W["up_proj"].T)) @ W["down_proj"].T

    def logits(self, x):
        return _unit(x, self.c["rms_norm_eps"]) * self.final @ self.head.T


class _Listed:
    """What the designs share whose layers are listed one by one (tensors of layer i start with ``l<i>.``)."""

    def __init__(self, config, get):
        self.c, self.layers, self.eps = config, len(config["layers"]), config["norm"]["eps"]
        self.all = [n for n in tensor_specs_for(dict(config))]
        self.embed, self.final = get("embed"), get("final.norm")
        self.final_bias = get("final.norm.b") if "final.norm.b" in self.all else None
        self.head = get("head") if "head" in self.all else self.embed
        self.pairs = get("bigram") if "bigram" in self.all else None

    def start(self, tokens):
        return self.embed[tokens]

    def names(self, i):
        return {n[len(f"l{i}."):]: n for n in self.all if n.startswith(f"l{i}.")}


class _Suranex(_Listed):
    def layer(self, i, W, x, tokens, memo):
        layer, eps = self.c["layers"][i], self.eps
        mixed = self.attention(W, layer["mixer"], x) if layer["type"] == "attention" else self.recurrence(W, layer["mixer"], x)
        x = x + _unit(mixed, eps) * (1.0 + W["norm1"])
        return x + _unit(self.experts(W, layer["mlp"], x, tokens), eps) * (1.0 + W["norm2"])

    def attention(self, W, m, h):
        n, eps, rot = h.shape[0], self.eps, m["rot"]
        q, k, v = ((h @ W["mix." + s].T).view(n, -1, m["dim"] if s != "v" else m["vdim"]) for s in "qkv")
        f, mag = _frequencies(rot["dims"], rot["base"], rot.get("scaling"), h.device)
        turned = _positions(n, f)
        q = _turn(_unit(q, eps) * W["mix.q.norm"], turned, "half", mag)
        k = _turn(_unit(k, eps) * W["mix.k.norm"], turned, "half", mag)
        by_value = _positions(n, _frequencies(m["vdim"], rot["base"], None, h.device)[0])
        v = _turn(_unit(v, eps), by_value, "half")
        at = torch.arange(n, device=h.device)
        near = (at[:, None] - at < m["mask"]["size"]) | (at < m["mask"]["keep_first"])
        o = _turn(_attend(q, k, v, m["scale"], m["softcap"], near & (at <= at[:, None])), -by_value, "half")
        o = o * torch.sigmoid(h @ W["mix.g"].T)[:, :, None]
        return o.reshape(n, -1) @ W["mix.o"].T

    def recurrence(self, W, m, h):
        n = h.shape[0]
        y = _gelu(h @ W["mix.y"].T + W["mix.y.b"])
        u = _convolution(h @ W["mix.x"].T + W["mix.x.b"], W["mix.conv"]) + W["mix.conv.b"]
        blocks = u.view(n, m["blocks"], -1)
        gate = lambda s: torch.sigmoid(torch.einsum("tbi,boi->tbo", blocks, W["mix." + s]) + W["mix." + s + ".b"]).reshape(n, -1)
        a = torch.exp(-8.0 * gate("ra") * torch.nn.functional.softplus(W["mix.lam"]))
        fed = torch.sqrt(1.0 - a * a) * gate("ri") * u
        state, out = torch.zeros_like(fed[0]), torch.empty_like(fed)
        for t in range(n):
            state = a[t] * state + fed[t]
            out[t] = state
        return (out * y) @ W["mix.o"].T

    def experts(self, W, f, h, tokens):
        def one(x, p, limit):
            g, u = (x @ W[p + "gate"].T).clamp(max=limit), (x @ W[p + "up"].T).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ W[p + "down"].T

        out, chosen = one(h, "mlp.shared.", f["shared"]["limit"]), W["mlp.table"].long()[tokens]
        for e in range(f["router"]["experts"]):
            rows = (chosen == e).any(1).nonzero()[:, 0]
            if rows.numel():
                out[rows] += one(h[rows], f"mlp.e{e}.", f["expert"]["limit"]) / f["router"]["top"]
        return out

    def logits(self, x):
        return _unit(x, self.eps) * (1.0 + self.final) @ self.head.T


class _Nutavik(_Listed):
    def norm(self, x, w, b):
        x = x - x.mean(-1, keepdim=True)
        return _unit(x, self.eps) * w + b

    def layer(self, i, W, x, tokens, memo):
        layer, mult = self.c["layers"][i], self.c["residual_mult"]
        norm = lambda x, s: self.norm(x, W[s], W[s + ".b"])
        h = norm(x, "norm1")
        if layer["type"] == "latent_attention":
            mixed = self.latent_attention(W, layer["mixer"], h, memo, i)
        else:
            o = self.delta(W, layer["mixer"], h) if layer["type"] == "delta" else self.linear(W, layer["mixer"], h)
            mixed = ((_unit(o, self.eps) * W["mix.norm"]).reshape(x.shape[0], -1) * _silu(h @ W["mix.g"].T)) @ W["mix.o"].T
        x = x + mult * norm(mixed, "norm1b")
        return x + mult * norm(torch.relu(norm(x, "norm2") @ W["mlp.up"].T) ** 2 @ W["mlp.down"].T, "norm2b")

    def latent_attention(self, W, m, h, memo, i):
        n, rank, rot = h.shape[0], m["kv_rank"], m["rot"]
        f, mag = _frequencies(rot["dims"], rot["base"], rot.get("scaling"), h.device)
        angle = _positions(n, f)
        q = ((_unit(h @ W["mix.dq"].T, self.eps) * W["mix.dq.norm"]) @ W["mix.uq"].T).view(n, m["heads"], -1)
        if m.get("kv_from") is None:
            both = h @ W["mix.dkv"].T
            memo[i] = _unit(both[:, :rank], self.eps) * W["mix.dkv.norm"], _turn(both[:, rank:], angle, "neighbours", mag)
        latent, turned = memo[i if m.get("kv_from") is None else m["kv_from"]]
        k = torch.cat([(latent @ W["mix.uk"].T).view(n, m["heads"], -1), turned[:, None].expand(n, m["heads"], -1)], -1)
        q = torch.cat([q[..., : m["dim"]], _turn(q[..., m["dim"]:], angle, "neighbours", mag)], -1)
        o = _attend(q, k, (latent @ W["mix.uv"].T).view(n, m["heads"], -1), m["scale"])
        return (o * torch.sigmoid(h @ W["mix.g"].T)[:, :, None]).reshape(n, -1) @ W["mix.o"].T

    def delta(self, W, m, h):
        z = torch.nn.functional.softplus(h @ W["mix.a"].T + W["mix.dt_bias"])
        return _delta_scan(W, m, h, torch.exp(-torch.exp(W["mix.A_log"]) * z)[:, :, None])

    def linear(self, W, m, h):
        n = h.shape[0]
        q, k, v = ((h @ W["mix." + s].T).view(n, m["heads"], -1) for s in "qkv")
        z = (h @ W["mix.a1"].T) @ W["mix.a2"].T + W["mix.a2.b"]
        keep = (torch.sigmoid(z) ** (1.0 / m["tau"])).view(n, m["heads"], -1, 1)
        state, out, q = torch.zeros(m["heads"], m["dim"], m["vdim"], dtype=F, device=h.device), torch.empty_like(v), q * m["dim"] ** -0.5
        for t in range(n):
            state = keep[t] * state + k[t][:, :, None] * v[t][:, None]
            out[t] = (q[t][:, None] @ state)[:, 0]
        return out

    def logits(self, x):
        return self.norm(x, self.final, self.final_bias) @ self.head.T * self.c["logit_scale"]


def _delta_scan(W, m, h, keep):
    """The delta rule; ``keep`` [n, heads, 1 or dim] is what a step leaves of the state's rows."""
    n, share = h.shape[0], m["heads"] // m["kv_heads"]
    q, k, v = (_silu(_convolution(h @ W["mix." + s].T, W["mix." + s + ".conv"])).view(n, -1, m["dim"] if s != "v" else m["vdim"]) for s in "qkv")
    length = lambda x: (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(share, 1)
    q, k, beta = length(q) * m["dim"] ** -0.5, length(k), torch.sigmoid(h @ W["mix.b"].T)
    state, out = torch.zeros(m["heads"], m["dim"], m["vdim"], dtype=F, device=h.device), torch.empty_like(v)
    for t in range(n):
        state = keep[t][:, :, None] * state
        lacks = beta[t][:, None] * (v[t] - (k[t][:, None] @ state)[:, 0])
        state = state + k[t][:, :, None] * lacks[:, None]
        out[t] = (q[t][:, None] @ state)[:, 0]
    return out


class _Rafusun(_Listed):
    def start(self, tokens):
        e = self.c["embedding"]
        b = e["bigram"]
        pair = torch.full_like(tokens, b["buckets"])
        pair[1:] = (tokens[:-1] * b["mul_prev"] + tokens[1:] * b["mul_cur"]) % b["buckets"]
        return self.embed[tokens] * e["scale"] + self.pairs[pair]

    def layer(self, i, W, x, tokens, memo):
        layer, alpha = self.c["layers"][i], self.c["postln_alpha"]
        m, n = layer["mixer"], x.shape[0]
        if layer["type"] == "channel_delta":
            z = (x @ W["mix.a1"].T) @ W["mix.a2"].T + W["mix.dt_bias"]
            z = torch.nn.functional.softplus(z).view(n, m["heads"], -1)
            o = _unit(_delta_scan(W, m, x, torch.exp(-torch.exp(W["mix.A_log"])[:, None] * z)), self.eps) * W["mix.norm"]
            gate = torch.sigmoid((x @ W["mix.g1"].T) @ W["mix.g2"].T)
            mixed = (o.reshape(n, -1) * gate) @ W["mix.o"].T
        else:
            left, right = self.attention(W, m["left"], x), self.time_mixing(W, m["right"], x)
            mixed = 0.5 * (_unit(left, self.eps) * W["mix.left.out"] + _unit(right, self.eps) * W["mix.right.out"])
        x = _unit(alpha * x + mixed * W["ls1"], self.eps) * W["norm1"]
        fed = (_gelu(x @ W["mlp.gate"].T) * (x @ W["mlp.up"].T)) @ W["mlp.down"].T
        return _unit(alpha * x + fed * W["ls2"], self.eps) * W["norm2"]

    def attention(self, W, m, h):
        n = h.shape[0]
        q, k, v = ((h @ W["mix.left." + s].T).view(n, -1, m["dim"] if s != "v" else m["vdim"]) for s in "qkv")
        angle = _positions(n, _frequencies(m["rot"]["dims"], m["rot"]["base"], None, h.device)[0])
        q, k = (_unit(_turn(s, angle, "neighbours"), self.eps) for s in (q, k))
        at = torch.arange(n, device=h.device)
        same = (at // m["mask"]["size"])[:, None] == at // m["mask"]["size"]
        return _attend(q, k, v, m["scale"], m["softcap"], same & (at <= at[:, None]), sink=True).reshape(n, -1) @ W["mix.left.o"].T

    def time_mixing(self, W, m, h):
        n, p = h.shape[0], "mix.right."
        past = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
        mix = lambda s: h + (past - h) * W[p + "mu." + s]
        r, k, v = ((mix(s) @ W[p + s].T).view(n, m["heads"], -1) for s in "rkv")
        z = torch.tanh(mix("w") @ W[p + "w1"].T) @ W[p + "w2"].T + W[p + "w0"]
        keep, now = torch.exp(-torch.exp(z)).view(n, m["heads"], -1, 1), W[p + "u"][:, :, None]
        state, out = torch.zeros(m["heads"], m["dim"], m["dim"], dtype=F, device=h.device), torch.empty_like(v)
        for t in range(n):
            written = k[t][:, :, None] * v[t][:, None]
            out[t] = (r[t][:, None] @ (state + now * written))[:, 0]
            state = keep[t] * state + written
        return (_unit(out, self.eps).reshape(n, -1) * W[p + "norm"] * _silu(mix("g") @ W[p + "g"].T)) @ W[p + "o"].T

    def logits(self, x):
        return _unit(x, self.eps) * self.final @ self.head.T


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "sample":
        return None  # a choice by a request's own stream of numbers: whole numbers, compared as they are
    config = _config(case)
    get = _weights(config, case["dtype"])
    plain = {"Suranex": _Suranex, "Nutavik": _Nutavik, "Rafusun": _Rafusun}.get(config.get("architecture"), _Llama)(config, get)
    tokens = [torch.tensor(s, device=plain.embed.device) for s in _sequences(case, seed)]
    streams, memos = [plain.start(t) for t in tokens], [{} for _ in tokens]
    for i in range(plain.layers):
        W = {short: get(name) for short, name in plain.names(i).items()}
        streams = [plain.layer(i, W, x, t, memo) for x, t, memo in zip(streams, tokens, memos)]
        del W
    out = []
    for step in _script(case)[0]:
        rows = [streams[r][first + w] for r, first, _, want in step for w in want]
        if rows:
            out.append(plain.logits(torch.stack(rows)))
    return out
